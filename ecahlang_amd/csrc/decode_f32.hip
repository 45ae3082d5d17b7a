// Paged decode over fp32 caches on the matrix cores (page_size 16, head_dim 64 or 128, GQA groups 1
// to 16).  Same contract as the vector kernel (BatchDecodeWithPagedKVCacheWrapper.run,
// ecahlang/main.py:68); everything stays in fp32: v_mfma_f32_16x16x4_f32 takes fp32 operands.
//
// A workgroup (W = 4 waves) takes one KV head of one part of one sequence's pages; wave r takes the part's
// pages r, r + W, ...  With lane l = (lr = l % 16, lg = l / 16), a page:
//   S[token][head]      = K . Q^T   A: lane holds K[token lr][dim 16 s + 4 lg + e], B: Q[head lr][the same
//                                   dims]: one 16-byte load feeds the four products e = 0 .. 3
//   online softmax                  lane: head lr, tokens 4 lg + i
//   O^T[dim][head]     += V^T . P   product i takes the tokens 4 lg + i, which are the lane's own softmax
//                                   weights: B is the score register itself.  A: V[token 4 lg + i][dim
//                                   64 c + 4 lr + e], one 16-byte load for the four output tiles e
// so K and V go from memory straight into the operand registers (no LDS, no lane exchange), each
// refilled with the next page's rows as soon as its products are issued, and the group's heads share
// every row read.  The waves' states meet in LDS at the end.  A sequence of several parts is merged by the
// workgroup that arrives last: of a KV head's parts, for that head, or (without head counters) of all of
// the sequence's, for all heads.
//
// What bounds it: the bytes of K and V at large batches (5.3 TB/s at 197 MB); a small batch is a chain
// of latencies (page list, page ids, rows: 5.2 us for one sequence of 100 tokens; partials, arrival,
// merge: 6 more).  Arrivals on one counter take their turns at the memory side, about 30 ns each, so
// every KV head of a sequence counts its own (16 sequences of 16 to 2048 tokens, 32 / 8 heads of 64
// dims: 16.8 us with one counter a sequence, 11.1 with one a head).  Four waves a workgroup rather than
// eight: more of them start while others wait (11.1 and 13.1 us).  On the vector kernel the same call
// took 280 us: every lane read a whole K row, V one token at a time, and a sequence of 2048 tokens was
// cut into 128 parts.  Error against 64 bits: 1.7e-7, 2.4e-7 there.
//
// A large batch of short sequences is bound by the workgroups there are, one per KV head and sequence
// (about 3.5 ns each): 1024 / 4096 / 8192 sequences of 16 tokens at 8 KV heads 30 / 110 / 235 us (65 / 266 /
// 571 on the vector kernel; 70 / 595 / 2071 when every workgroup looked through the whole batch for its
// part).  Below about four tokens a sequence the vector kernel's few workgroups are still ahead there (16 KV
// heads, 1024 sequences of 1 / 4 / 16 tokens: 48 us for its 28 / 43 / 103); the host does not know the lengths.
#include <algorithm>
#include "attn_common.h"
#include "mfma_common.h"

using namespace pkv;
using namespace pkv::mfma;

namespace {

constexpr int W = 4;               // waves per workgroup
constexpr int kMinPages = 8;       // pages per part of a cut sequence, about, at least (16: 12.9 us for 11.1 at
                                   // 16 sequences of 16 to 2048 tokens; 4: 21.6 for 16.8, one counter a sequence)
constexpr float kLazyMax = 8.f;    // a head's reference max moves only on jumps > 2^8
constexpr int kMergeParts = 16;    // parts whose rows the merge loads at a time

// Parts of a sequence of np pages (np 0: one, which writes zeros), of about `aim` pages each,
// max_parts at most.
__device__ __forceinline__ int parts_of(int np, int aim, int max_parts) {
  return max(min((np + aim - 1) / aim, max_parts), 1);
}

template <int D, bool APP>
__global__ __launch_bounds__(W * 64, D == 64 ? 4 : 2) void decode_f32_kernel(DecodeParams P, int nr, int max_parts, int head_counters) {
  constexpr int QS = D / 16;  // 16-dim pieces of a row
  constexpr int NC = D / 64;  // 64-dim pieces of the output
  constexpr int NP = NC * 4;  // 16-byte pieces of a lane's 16 NC output values
  __shared__ f4 s_o[W][NP][64];
  __shared__ float2 s_ml[W][16];
  __shared__ int s_last;

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int B = P.batch, g = P.hq / P.hkv;
  const int h = blockIdx.x % P.hkv, w = blockIdx.x / P.hkv;

  // ---- workgroup w: the first part of sequence w, or (w >= B) the (w - B)-th of the further parts, which
  // follow each other in sequence order.  Only those and cut sequences look for their place among the
  // batch, 64 sequences a round (each workgroup over all of it, the time of a large batch of short
  // sequences went with its square).
  const int cut = (int)min((int64_t)INT_MAX, P.num_indices);  // the page list ends there
  const int own = min(w, B - 1);
  int ip0 = P.indptr[min(lane, B)], ip1 = P.indptr[min(lane + 1, B)], lastv = P.last[min(lane, B - 1)];
  int b = own, s0 = P.indptr[own], e0 = P.indptr[own + 1], lastp = P.last[own];
  const int total = max(min(P.indptr[B], cut), 1);
  const int aim = max(kMinPages, (total + nr - 1) / nr);
  auto listed = [&](int i0, int i1) { return max(min(i1, cut) - max(i0, 0), 0); };  // pages of the list
  int avail = listed(s0, e0), nparts = parts_of(avail, aim, max_parts), part = 0, more0 = 0;
  if (w >= B || nparts > 1) {
    bool found = false;
    int base = 0;
#pragma unroll 1
    for (int b0 = 0; b0 < B; b0 += 64) {
      const int n0 = P.indptr[min(b0 + 64 + lane, B)], n1 = P.indptr[min(b0 + 65 + lane, B)];  // (the next round's)
      const int nl = P.last[min(b0 + 64 + lane, B - 1)];
      const int av = listed(ip0, ip1);
      const int n = b0 + lane < B ? parts_of(av, aim, max_parts) - 1 : 0;
      int incl = n;
#pragma unroll
      for (int x = 1; x < 64; x <<= 1) {
        const int v = __shfl_up(incl, x, 64);
        incl += lane >= x ? v : 0;
      }
      const int all = __builtin_amdgcn_readlane(incl, 63);
      if (w < B ? w < b0 + 64 : w - B < base + all) {
        const int l = w < B ? w - b0 : __popcll(__ballot(base + incl <= w - B));
        more0 = base + __builtin_amdgcn_readlane(incl, l) - __builtin_amdgcn_readlane(n, l);
        if (w >= B) {
          b = b0 + l;
          s0 = __builtin_amdgcn_readlane(ip0, l);
          e0 = __builtin_amdgcn_readlane(ip1, l);
          lastp = __builtin_amdgcn_readlane(lastv, l);
          avail = __builtin_amdgcn_readlane(av, l);
          nparts = parts_of(avail, aim, max_parts);
          part = 1 + w - B - more0;
        }
        found = true;
        break;
      }
      base += all;
      ip0 = n0, ip1 = n1, lastv = nl;
    }
    if (!found) return;  // (the grid is sized for the most parts there can be)
    nparts = 1 + min(nparts - 1, max(nr - more0, 0));  // (a kv_indptr that runs backwards)
  }
  const int np = e0 - s0;
  // the part's pages [p0, end) of the page list, a wave's p0 + wave, + W, ... (the ids of 64 of them a
  // lane each)
  const int per = avail / nparts, more = avail - per * nparts;  // (the first `more` parts hold a page more)
  const int p0 = max(s0, 0) + part * per + min(part, more), end = p0 + per + (part < more ? 1 : 0);
  const int len = np > 0 ? (np - 1) * 16 + lastp : 0;
  const int n = end - p0 > wave ? (end - p0 - 1 - wave) / W + 1 : 0;
  // a sequence of one page at most is wave 0's, which writes its own state; the others leave their
  // places to further workgroups
  const bool one = nparts == 1 && end - p0 <= 1;
  if (one && wave > 0) return;
  int pidv = n > 0 ? P.indices[min(p0 + wave + W * lane, end - 1)] : -1;

  const int64_t rowstride = (int64_t)P.hkv * D, hoff = (int64_t)h * D;
  const float* kc = reinterpret_cast<const float*>(P.k_cache) + hoff + lr * rowstride + 4 * lg;
  const float* vc = reinterpret_cast<const float*>(P.v_cache) + hoff + 4 * lg * rowstride + 4 * lr;
  // columns past the group repeat its last head (never stored)
  const float* qc = reinterpret_cast<const float*>(P.q) + (int64_t)(h * g + (lr < g ? lr : g - 1)) * P.q_sh + 4 * lg;
  // (global address space by name: a store through a generic pointer makes the compiler drain every
  // load in flight at the waits that follow)
  typedef __attribute__((address_space(1))) float gfloat;
  gfloat* out = (gfloat*)P.out;
  const bool o16 = (((uintptr_t)P.out | (uintptr_t)(P.o_sn * 4) | (uintptr_t)(P.o_sh * 4)) & 15) == 0;

  // The step's new token (pkv_batch_decode_append) goes to the sequence's last position: page app_pi of
  // the page list, row app_row.  Its rows are loaded in place of that row of the page, and stored there
  // once they are in (one wave of one workgroup loads the page for this KV head).  A launch of its own
  // for it costs 3 us more a call (18.9 and 21.8).  APP keeps its selects out of calls without one (0.6 us).
  const bool app = APP && s0 >= 0 && np > 0 && avail == np && lastp >= 0 && lastp <= 16 && len > 0;
  const int app_pi = app ? s0 + (len - 1) / 16 : -1, app_row = (len - 1) & 15;
  const float* akp = app ? reinterpret_cast<const float*>(P.ak + b * P.ak_sn + h * P.ak_sh) + 4 * lg : nullptr;
  const float* avp = app ? reinterpret_cast<const float*>(P.av + b * P.av_sn + h * P.av_sh) + 4 * lr : nullptr;

  // Rows of page k of this wave.  The loads are unconditional, so that every path has the same ones
  // in flight and the waits stay exact: past the wave's last page, and for an id outside the pool,
  // they read a query row instead.
  f4 kr[QS], vr[4][NC];
  auto page_of = [&](int k) __attribute__((always_inline)) -> int {
    const int pid = __builtin_amdgcn_readlane(pidv, k & 63);
    return k < n && pid >= 0 && (int64_t)pid < P.num_pages ? pid : -1;
  };
  const float* const dummy = qc - 4 * lg;
  auto load_k = [&](int pid, int pi) __attribute__((always_inline)) {
    const float* kp = pid >= 0 ? kc + pid * P.page_stride : dummy;
    if (APP) kp = pid >= 0 && pi == app_pi && lr == app_row ? akp : kp;
#pragma unroll
    for (int s = 0; s < QS; ++s) kr[s] = *reinterpret_cast<const f4*>(kp + 16 * s);
  };
  auto load_v = [&](int pid, int pi) __attribute__((always_inline)) {
    const float* vp = pid >= 0 ? vc + pid * P.page_stride : dummy;
    const int64_t rs = pid >= 0 ? rowstride : 0;
    const int ar = APP && pid >= 0 && pi == app_pi ? app_row - 4 * lg : -1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float* rp = APP && i == ar ? avp : vp + i * rs;
#pragma unroll
      for (int c = 0; c < NC; ++c) vr[i][c] = *reinterpret_cast<const f4*>(rp + 64 * c);
    }
  };
  int k = 0, pid = page_of(0);
  load_k(pid, p0 + wave);
  load_v(pid, p0 + wave);

  f4 qr[QS];  // in base-2 units
#pragma unroll
  for (int s = 0; s < QS; ++s) qr[s] = *reinterpret_cast<const f4*>(qc + b * P.q_sn + 16 * s) * P.scale_log2;
  f4 o[NC][4];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) o[c][e] = f4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;

#pragma unroll 1
  for (int pi = p0 + wave; pi < end; pi += W) {
    f4 sa = f4{0.f, 0.f, 0.f, 0.f}, sb = sa;  // (two chains: a product waits for the one two back)
#pragma unroll
    for (int s = 0; s < QS; ++s)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        sa = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[s][e], qr[s][e], sa, 0, 0, 0);
        sb = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[s][e + 1], qr[s][e + 1], sb, 0, 0, 0);
      }
    const int left = len - 16 * (pi - s0);
    const int nv = pid < 0 || left < 0 ? 0 : left;  // tokens of the page that exist (16 and above: all)
    if (APP && pi == app_pi && pid >= 0) {
      typedef __attribute__((address_space(1))) f4 gf4;
      if (lr == app_row) {
#pragma unroll
        for (int s = 0; s < QS; ++s) *(gf4*)(kc + pid * P.page_stride + 16 * s) = kr[s];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (4 * lg + i == app_row) {
#pragma unroll
          for (int c = 0; c < NC; ++c) *(gf4*)(vc + pid * P.page_stride + i * rowstride + 64 * c) = vr[i][c];
        }
    }
    ++k;
    if ((k & 63) == 0) {
      pidv = P.indices[min(pi + W * (1 + lane), end - 1)];
      __builtin_amdgcn_s_waitcnt(0x0F70);  // (compiler-visible vmcnt(0): the usual path waits for nothing)
    }
    pid = page_of(k);
    load_k(pid, pi + W);
    sa += sb;
    if (nv < 16) {
      // tokens past the sequence's end: no score, and rows read as zeros (0 * NaN would poison P.V)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool in = 4 * lg + i < nv;
        sa[i] = in ? sa[i] : -INFINITY;
#pragma unroll
        for (int c = 0; c < NC; ++c) vr[i][c] = in ? vr[i][c] : f4{0.f, 0.f, 0.f, 0.f};
      }
    }
    const float cms = max_across_groups(max2f(max2f(sa[0], sa[1]), max2f(sa[2], sa[3])));
    const bool grow = cms > m + kLazyMax;  // (false while every score so far is -inf)
    if (__ballot(grow)) {
      const float mnew = grow ? cms : m;
      // 0 from -inf; 1 if unchanged (also where no score has been seen: -inf less -inf is NaN)
      const float alpha = grow ? __builtin_amdgcn_exp2f(m - mnew) : 1.f;
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[c][e] *= alpha;
      lsum *= alpha;
      m = mnew;
    }
    const float nm = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int i = 0; i < 4; ++i) sa[i] = __builtin_amdgcn_exp2f(sa[i] - nm);
    lsum += (sa[0] + sa[1]) + (sa[2] + sa[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[c][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[i][c][e], sa[i], o[c][e], 0, 0, 0);
    load_v(pid, pi + W);
  }

  // ---- the waves' states in wave order (a wave without a page: no mass)
  const float ltot = sum_across_groups(lsum);
  if (lg == 0) s_ml[wave][lr] = make_float2(m, ltot);
  lds_barrier();
  float2 v[W];
#pragma unroll
  for (int x = 0; x < W; ++x) v[x] = x == 0 || !one ? s_ml[x][lr] : make_float2(-INFINITY, 0.f);
  float M = -INFINITY, L = 0.f;
#pragma unroll
  for (int x = 0; x < W; ++x) M = fmaxf(M, v[x].x);
  const float mu = M == -INFINITY ? 0.f : M;
#pragma unroll
  for (int x = 0; x < W; ++x) L += v[x].y * __builtin_amdgcn_exp2f(v[x].x - mu);
  const float cs = __builtin_amdgcn_exp2f(m - mu);
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i)  // dims 64 c + 16 lg + 4 i + (0 .. 3)
      s_o[wave][4 * c + i][lane] = f4{o[c][0][i], o[c][1][i], o[c][2][i], o[c][3][i]} * cs;
  lds_barrier();
  auto store_row = [&](int64_t hq, int d, f4 x) __attribute__((always_inline)) {
    gfloat* dst = out + b * P.o_sn + hq * P.o_sh + d;
    if (o16) {
      *(__attribute__((address_space(1))) f4*)dst = x;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) dst[e] = x[e];
    }
  };
  if (lr < g) {
    const float inv = L > 0.f ? 1.f / L : 0.f;
    const int64_t hq = h * g + lr;
#pragma unroll 1
    for (int pc = wave; pc < NP; pc += one ? 1 : W) {  // piece 4 c + i by wave (4 c + i) % W
      f4 acc = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int x = 0; x < W; ++x) {
        const f4 y = s_o[x][pc][lane];
        acc += x == 0 || !one ? y : f4{0.f, 0.f, 0.f, 0.f};
      }
      acc *= inv;
      const int d = 64 * (pc / 4) + 16 * lg + 4 * (pc % 4);
      if (nparts == 1) store_row(hq, d, acc);
      else st_dev4(P.part_o, (uint32_t)((((int64_t)w * P.hq + hq) * D + d) * sizeof(float)), acc);
    }
    if (nparts > 1 && wave == 0 && lg == 0) store_partial_ml(P, w, (int)hq, M, L);
  }
  if (nparts == 1) return;
  if (!arrive_last(P, head_counters ? b * P.hkv + h : b, head_counters ? nparts : nparts * P.hkv, &s_last)) return;

  // ---- merge of the sequence's parts, for this KV head or (one counter a sequence) for all: four dims
  // of one head a lane, the parts shared by nw waves, the rows of kMergeParts parts requested at once
  // and folded under a running max (a part without mass holds zeros; repeats weigh nothing).  With head
  // counters a line of (max, sum) pairs has a reader per KV head, so the pairs are loaded past the
  // caches (ld_dev2); a head's partial rows are whole lines of its own.
  const int x0 = head_counters ? h * g * (D / 4) : 0, nx = (head_counters ? g : P.hq) * (D / 4);
  const int groups = (nx + 63) / 64, nw = groups >= W ? 1 : W / groups;  // waves a group of 64 items
  const int share = (nparts + nw - 1) / nw;
  for (int gr = wave / nw; gr < (groups + W / nw - 1) / (W / nw) * (W / nw); gr += W / nw) {  // (the same rounds for every wave)
    const int x = x0 + min(gr * 64 + lane, nx - 1);
    const int hq = x / (D / 4), d = (x - hq * (D / 4)) * 4;
    const float2* ml = P.part_ml + hq;
    const float* po = P.part_o + (int64_t)hq * D + d;
    const int q1 = min(share * (wave % nw + 1), nparts);
    float M2 = -INFINITY, den = 0.f;
    f4 acc = f4{0.f, 0.f, 0.f, 0.f};
    auto fold = [&](float mx, float l, f4 row, float mn) __attribute__((always_inline)) {
      const float c = __builtin_amdgcn_exp2f(mx - mn) * l;
      den += c;
      acc += c * row;
    };
    for (int q0 = share * (wave % nw); q0 < q1; q0 += kMergeParts) {
      float2 y[kMergeParts];
      f4 row[kMergeParts];
#pragma unroll
      for (int q = 0; q < kMergeParts; ++q) {
        const int pq = min(q0 + q, q1 - 1);
        const int64_t sl = pq == 0 ? b : B + more0 + pq - 1;
        y[q] = ld_dev2(ml + sl * P.ml_stride);
        row[q] = *reinterpret_cast<const f4*>(po + sl * P.hq * D);
      }
      float Mn = M2;
#pragma unroll
      for (int q = 0; q < kMergeParts; ++q) Mn = fmaxf(Mn, y[q].x);
      const float mn = Mn == -INFINITY ? 0.f : Mn, f = __builtin_amdgcn_exp2f(M2 - mn);
      den *= f;
      acc *= f;
      M2 = Mn;
#pragma unroll
      for (int q = 0; q < kMergeParts; ++q)
        if (q0 + q < q1) fold(y[q].x, y[q].y, row[q], mn);
    }
    if (nw > 1) {  // (then every group is a round of its own)
      __syncthreads();
      s_o[wave][0][lane] = acc;
      s_o[wave][1][lane] = f4{M2, den, 0.f, 0.f};
      __syncthreads();
      if (wave % nw != 0) continue;
      float Mn = -INFINITY;
      for (int y = 0; y < nw; ++y) Mn = fmaxf(Mn, s_o[wave + y][1][lane][0]);
      const float mn = Mn == -INFINITY ? 0.f : Mn;
      acc = f4{0.f, 0.f, 0.f, 0.f};
      den = 0.f;
      for (int y = 0; y < nw; ++y) {
        const f4 z = s_o[wave + y][1][lane];
        const float f = __builtin_amdgcn_exp2f(z[0] - mn);
        den += f * z[1];
        acc += f * s_o[wave + y][0][lane];
      }
    }
    if (gr * 64 + lane < nx) store_row(hq, d, acc * (den > 0.f ? 1.f / den : 0.f));
  }
}

}  // namespace

namespace pkv {

bool decode_f32_supported(int dtype, int d, int g, int ps) {
  return dtype == kF32 && (d == 64 || d == 128) && g >= 1 && g <= 16 && ps == 16;
}

int decode_f32_dispatch(const DecodeParams& P, int d, bool head_counters, hipStream_t s) {
  // Parts are sized for 3/4 of num_ctas / 2 CUs x 4 workgroups (2 at head_dim 128): the parts that
  // sequences of unequal lengths round up to then start in about one wave of workgroups.  32 / 8 heads
  // of 64 dims, 64 sequences of 20 to 700 tokens / 40 of 1200, in us: 1/2 18.0 / 37.7, 3/4 18.1 / 37.1,
  // 1 19.8 / 38.3, 4 19.9 / 41.6; 16 / 2 of 128, 64 of 100 to 1500: 28.7, 24.5, 28.1, 28.1.  (nr + batch
  // parts at most; the workspace has slots for num_ctas + batch.)
  const int64_t want = (int64_t)(d == 64 ? 6 : 3) * P.num_ctas / (4 * P.hkv);
  const int nr = (int)std::max<int64_t>(std::min<int64_t>(P.num_ctas, want), 1);
  const int max_parts = std::max(64, P.num_ctas / P.hkv);
  const int64_t wgs = ((int64_t)nr + P.batch) * P.hkv;
  if (wgs > INT32_MAX) return kBadArg;
  const dim3 grid((unsigned)wgs);
#define PKV_DECODE_F32(D, APP)                                                                               \
  hipLaunchKernelGGL((decode_f32_kernel<D, APP>), grid, dim3(W * 64), 0, s, P, nr, max_parts, head_counters ? 1 : 0)
  if (d == 64) {
    if (P.ak) PKV_DECODE_F32(64, true);
    else PKV_DECODE_F32(64, false);
  } else {
    if (P.ak) PKV_DECODE_F32(128, true);
    else PKV_DECODE_F32(128, false);
  }
#undef PKV_DECODE_F32
  return (int)hipGetLastError();
}

}  // namespace pkv
