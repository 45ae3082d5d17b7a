// Top-k / top-p sampling from logits, the sampler the serving loop calls after the last layer
// (flashinfer.sampling.top_k_top_p_sampling_from_logits at
// ecahlang/main.py:377-379, 400-402, 489-491, 582-584; top-k filter first, then top-p on the
// renormalised top-k distribution, deterministic=True).
//
// Definition (the oracle, oracle/sampling_ref.py, restates the same rule):
//   p_i ∝ exp(x_i - max x)                                   (softmax of the row's logits)
//   K   = { i : x_i >= k-th largest logit }                  (all tokens when k <= 0 or k >= V)
//   S   = { i in K : x_i >= t }, t the largest logit with mass({j in K : x_j >= t}) >= top_p * mass(K)
//                                                             (S = K when top_p >= 1)
//   token = first i in S, in vocabulary order, whose cumulative mass over S exceeds u * mass(S)
// Ties at a threshold are kept.  No sort, and every mass is an integer: exp(x_i - max) in 32-bit fixed
// point, summed in 64 bits, so the result depends on nothing but the row and u (no floating-point
// summation order), nor on which of two ways a row goes:
//   one workgroup (sample_kernel: top-k filters over kTopKMax with any top-p, rows that the other kernels
//   hand back, calls without a workspace): both thresholds by radix selection over an order-preserving
//   32-bit key of the logit (three digit passes of 11, 11 and 10 bits, histograms in LDS).  Every pass reads
//   the row with 16-byte loads (8 fp16/bf16 or 4 fp32 logits per thread, 8 tiles in flight); after the first
//   one the row is served from L2.
//   many workgroups (the split kernels): all other rows, cut into slices.
#include <type_traits>
#include "common.h"
#include "../../include/pagedkv.h"

using namespace pkv;

namespace {

constexpr int kThreads = 1024;
constexpr int kBins = 2048;        // 11-bit digits
constexpr int kMaxTiles = 512;     // tiles of kThreads * 8 logits: vocabularies up to 4 M


// Order-preserving key of a float (larger float, larger key); NaN sorts lowest.
__device__ __forceinline__ uint32_t fkey(float f) {
  const uint32_t b = __float_as_uint(f);
  if (f != f) return 0u;
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
// The float whose fkey is k (k != 0).
__device__ __forceinline__ float key_float(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
// Mass of a logit in 32-bit fixed point: floor(exp(x - max) * 2^32), capped at 4294967040 (the
// largest float below 2^32), so it converts with one 32-bit instruction (a float -> 64-bit
// integer conversion is a sequence of ten; this runs for every logit on several passes).
__device__ __forceinline__ uint64_t fmass(float x, float mx) {
  const float d = x - mx;
  if (!(d > -23.f)) return 0;  // (also NaN): exp(-23) * 2^32 < 0.5
  return (uint64_t)(uint32_t)fminf(__expf(d) * 4294967296.0f, 4294967040.0f);
}

template <typename T>
struct Row {
  const T* p;
  int v;
  bool vec;
  static constexpr int E = 16 / sizeof(T);  // logits per 16-byte load
  // Calls f(index, logit) for this thread's logits of tile `tile` (thread t: E consecutive).
  template <typename F>
  __device__ __forceinline__ void tile(int tile, F&& f) const {
    const int base = (tile * kThreads + (int)threadIdx.x) * E;
    if (vec && base + E <= v) {
      const uint4 u = *reinterpret_cast<const uint4*>(p + base);
      const T* e = reinterpret_cast<const T*>(&u);
#pragma unroll
      for (int k = 0; k < E; ++k) f(base + k, to_f32(e[k]));
    } else {
#pragma unroll
      for (int k = 0; k < E; ++k)
        if (base + k < v) f(base + k, to_f32(p[base + k]));
    }
  }
  __device__ __forceinline__ int tiles() const { return (v + kThreads * E - 1) / (kThreads * E); }
  // Calls f(index, logit) for all of this thread's logits, kUnroll tiles' loads in flight at a time.
  static constexpr int kUnroll = 8;
  template <typename F>
  __device__ __forceinline__ void each(F&& f) const {
    const int nt = tiles();
    // (unconditional loads from clamped addresses: a load under a branch would be waited for
    // at the branch's end, one at a time; whole vectors past the row end are never used)
    const int last = v >= E ? (v - E) / E * E : 0;
    for (int t0 = 0; t0 < nt; t0 += kUnroll) {
      uint4 buf[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const int base = ((t0 + u) * kThreads + (int)threadIdx.x) * E;
        buf[u] = vec ? *reinterpret_cast<const uint4*>(p + min(base, last)) : make_uint4(0, 0, 0, 0);
      }
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const int base = ((t0 + u) * kThreads + (int)threadIdx.x) * E;
        if (vec && base + E <= v) {
          const T* e = reinterpret_cast<const T*>(&buf[u]);
#pragma unroll
          for (int k = 0; k < E; ++k) f(base + k, to_f32(e[k]));
        } else {
          for (int k = 0; k < E; ++k)
            if (base + k < v) f(base + k, to_f32(p[base + k]));
        }
      }
    }
  }
};

__device__ __forceinline__ float block_max(float v, float* red) {
  v = wave_max_f32(v);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) red[w] = v;
  __syncthreads();
  float r = -INFINITY;
  for (int i = 0; i < kThreads / 64; ++i) r = fmaxf(r, red[i]);
  return r;
}
__device__ __forceinline__ uint32_t block_max_u32(uint32_t v, uint32_t* red) {
  v = wave_max_u32(v);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) red[w] = v;
  __syncthreads();
  uint32_t r = 0;
  for (int i = 0; i < kThreads / 64; ++i) r = max(r, red[i]);
  return r;
}
__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) { return wave_sum_u64_dpp(v); }
__device__ __forceinline__ uint64_t block_sum_u64(uint64_t v, uint64_t* red) {
  v = wave_sum_u64(v);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) red[w] = v;
  __syncthreads();
  uint64_t r = 0;
  for (int i = 0; i < kThreads / 64; ++i) r += red[i];
  return r;
}

// What the launches over many workgroups leave of a row they hand back (fallback[row]): nothing but the
// row, the range of keys that holds the k-th largest (known.above .. known.need), or the bin that holds the
// top-p threshold.
enum Back : int { kNotBack = 0, kBackRow = 1, kBackKeys = 2, kBackBin = 3 };
constexpr int kPBins = 1024;  // bins of a top-p row's mass
// Where a top-p row's threshold lies: its bin (-1: no mass), the mass of the bins above it, the mass to
// reach.
struct ToppBin {
  uint64_t above, need;
  float mx, scale;  // (PBins)
  int64_t bin;
};
struct PBins {
  float mx, scale;
  __device__ __forceinline__ PBins(float mx_, float scale_) : mx(mx_), scale(scale_) {}
  __device__ __forceinline__ PBins(float2 range)
      : mx(range.x), scale((float)kPBins / fmaxf(fminf(range.x - range.y, 23.f), 1e-20f)) {}
  __device__ __forceinline__ int of(float x) const { return min((int)((mx - x) * scale), kPBins - 1); }
  // The finer bin of a logit of bin b.
  __device__ __forceinline__ int finer(float x, int b) const {
    return min((int)(__builtin_fmaf(mx - x, scale, -(float)b) * (float)kPBins), kPBins - 1);
  }
};

struct SampleLds {
  uint64_t hist[kBins];     // counts (top-k) or masses (top-p) per digit
  uint64_t tile[kMaxTiles];  // kept mass per tile
  uint64_t tile2[kMaxTiles];  // (row_from_bin: mass in the finer bin; the candidates' masses)
  uint64_t red[kThreads / 64];
  float redf[kThreads / 64];
  uint64_t scan[kThreads / 64];
  uint32_t sel[4];
};

// The bins of a row whose masses are in L.hist[0 .. kPBins): the one at which the mass from the first one on,
// `above` included, reaches need; above becomes the mass before it.
__device__ __forceinline__ int mass_bin(SampleLds& L, uint64_t& above, uint64_t need) {
  static_assert(kPBins == kThreads, "a bin a thread");
  const int t = threadIdx.x;
  const uint64_t own = L.hist[t];
  uint64_t upto = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t v = __shfl_up(upto, o, kWave);
    if ((t & 63) >= o) upto += v;
  }
  if ((t & 63) == 63) L.scan[t >> 6] = upto;
  __syncthreads();
  upto += above;
  for (int i = 0; i < t >> 6; ++i) upto += L.scan[i];
  if (upto >= need && upto - own < need) {
    L.sel[0] = t;
    L.sel[1] = (uint32_t)(upto - own);
    L.sel[2] = (uint32_t)((upto - own) >> 32);
  }
  __syncthreads();
  above = (uint64_t)L.sel[1] | (uint64_t)L.sel[2] << 32;
  return (int)L.sel[0];
}

// A top-p row whose bin is known but holds more logits than split_finish_kernel takes.  One pass over the row
// for the bin's mass in finer bins and its range of keys: mostly they are alike (ties are why there are so
// many), and that is the threshold.  Else a second takes the tiles' mass before the finer bin that the target
// falls in, and that bin's logits, among which the threshold is found (tiles: the tiles' kept masses are in
// L.tile).  False if there are too many of them.  (128 rows of 151,936 logits in steps of 1/4: 113 us a call,
// 223 when such rows started over, 151 when all top-p rows ran on one workgroup.)
template <typename RowT>
__device__ __forceinline__ bool row_from_bin(const RowT& row, SampleLds& L, const ToppBin& tb, uint32_t& thr, bool& tiles) {
  constexpr int kPairs = 256;  // keys compared each with all
  const PBins bins(tb.mx, tb.scale);
  const int t = threadIdx.x, cb = (int)tb.bin;
  tiles = false;
  L.hist[t] = 0;
  __syncthreads();
  uint32_t kmax = 0, knot = 0;  // largest key and (complemented) smallest
  row.each([&](int, float x) {
    if (bins.of(x) != cb) return;
    const uint64_t f = fmass(x, tb.mx);
    if (f) {
      atomicAdd((unsigned long long*)&L.hist[bins.finer(x, cb)], (unsigned long long)f);
      kmax = max(kmax, fkey(x));
      knot = max(knot, ~fkey(x));
    }
  });
  kmax = block_max_u32(kmax, reinterpret_cast<uint32_t*>(L.red));  // (and the finer bins are complete)
  knot = block_max_u32(knot, reinterpret_cast<uint32_t*>(L.red));
  thr = kmax;
  if (kmax == ~knot) return true;  // (uniform)
  tiles = true;
  uint64_t above = tb.above;
  const int fb = mass_bin(L, above, tb.need);
  const int ntiles = row.tiles();
  for (int i = t; i < ntiles; i += kThreads) L.tile[i] = L.tile2[i] = 0;
  if (t == 0) L.sel[3] = 0;
  __syncthreads();  // (and every thread has read the finer bins)
  kmax = knot = 0;
  uint64_t m = 0, m2 = 0;
  int cur = 0;
  auto flush = [&]() __attribute__((always_inline)) {
    if (m) atomicAdd((unsigned long long*)&L.tile[cur], (unsigned long long)m);
    if (m2) atomicAdd((unsigned long long*)&L.tile2[cur], (unsigned long long)m2);
    m = m2 = 0;
  };
  row.each([&](int i, float x) {
    const int tile = i / (kThreads * RowT::E);
    if (tile != cur) {  // (tiles come in increasing order)
      flush();
      cur = tile;
    }
    const int bin = bins.of(x);
    if (bin > cb) return;
    const uint64_t f = fmass(x, tb.mx);
    const int fi = bin < cb ? -1 : bins.finer(x, cb);
    m += fi < fb ? f : 0;
    if (fi == fb && f) {
      m2 += f;
      const uint32_t key = fkey(x), pos = atomicAdd(&L.sel[3], 1u);
      if (pos < kBins) L.hist[pos] = (uint64_t)(uint32_t)i << 32 | key;
      kmax = max(kmax, key);
      knot = max(knot, ~key);
    }
  });
  flush();
  kmax = block_max_u32(kmax, reinterpret_cast<uint32_t*>(L.red));  // (and the candidates are written)
  knot = block_max_u32(knot, reinterpret_cast<uint32_t*>(L.red));
  const int n = (int)L.sel[3];
  thr = kmax;
  if (kmax == ~knot) {
    for (int i = t; i < ntiles; i += kThreads) L.tile[i] += L.tile2[i];
    __syncthreads();
    return true;
  }
  if (n > kBins) return false;
  if (n <= kPairs) {
    // the largest key that enough mass reaches: each against all
    if (t < n) L.tile2[t] = fmass(key_float((uint32_t)L.hist[t]), tb.mx);
    __syncthreads();
    const uint32_t key = (uint32_t)L.hist[min(t, n - 1)];
    uint64_t sum = above;
    for (int i = 0; i < n; ++i) sum += (uint32_t)L.hist[i] >= key ? L.tile2[i] : 0;
    thr = block_max_u32(sum >= tb.need ? key : 0u, reinterpret_cast<uint32_t*>(L.red));
  } else {
    // the largest value that it reaches: of the bits in which the keys differ, from the highest
    uint32_t bit = 0x80000000u >> __builtin_clz(kmax ^ ~knot);
    for (thr = kmax & ~(2 * bit - 1); bit; bit >>= 1) {
      uint64_t sum = 0;
      for (int i = t; i < n; i += kThreads) {
        const uint32_t key = (uint32_t)L.hist[i];
        sum += key >= (thr | bit) ? fmass(key_float(key), tb.mx) : 0;
      }
      if (above + block_sum_u64(sum, L.red) >= tb.need) thr |= bit;
    }
  }
  for (int i = t; i < n; i += kThreads) {
    const uint32_t key = (uint32_t)L.hist[i];
    if (key >= thr)
      atomicAdd((unsigned long long*)&L.tile[(uint32_t)(L.hist[i] >> 32) / (kThreads * RowT::E)],
                (unsigned long long)fmass(key_float(key), tb.mx));
  }
  __syncthreads();
  return true;
}

template <typename T, typename RowT>
__device__ __forceinline__ void sample_row(const RowT& row, SampleLds& L, int b, int vocab, const int32_t* top_k,
                                           int32_t top_k_all, const float* top_p, float top_p_all,
                                           const float* uniform, int32_t* out, int how, const ToppBin* known) {
  uint64_t* s_hist = L.hist;
  uint64_t* s_tile = L.tile;
  uint64_t* s_red = L.red;
  float* s_redf = L.redf;
  uint64_t* s_scan = L.scan;
  uint32_t* s_sel = L.sel;
  uint32_t* s_sel32 = reinterpret_cast<uint32_t*>(L.red);
  const int ntiles = row.tiles();

  // ---- max logit; in a range of keys that holds the k-th largest, whether all are alike
  float mx = -INFINITY;
  uint32_t thr = 0;
  bool have_k = false;
  if (how == kBackKeys) {
    const uint32_t lo = (uint32_t)known->above, hi = (uint32_t)known->need;
    uint32_t kmax = 0, knot = 0;  // largest key and (complemented) smallest
    row.each([&](int, float x) {
      mx = fmaxf(mx, x);
      const uint32_t key = fkey(x);
      if (key >= lo && key <= hi) {
        kmax = max(kmax, key);
        knot = max(knot, ~key);
      }
    });
    kmax = block_max_u32(kmax, s_sel32);
    knot = block_max_u32(knot, s_sel32);
    have_k = kmax == ~knot;
    thr = have_k ? kmax : 0u;
  } else if (how != kBackBin) {
    row.each([&](int, float x) { mx = fmaxf(mx, x); });
  }
  mx = how == kBackBin ? known->mx : block_max(mx, s_redf);
  bool have_tiles = false;
  const bool have_p = how == kBackBin && row_from_bin(row, L, *known, thr, have_tiles);
  have_tiles = have_tiles && have_p;
  if (!have_k && !have_p) thr = 0;

  // ---- radix selection, most significant digit first.  `above` is what lies above the
  // current prefix (a count for top-k, a mass for top-p); the digit where the running total
  // from the top reaches `need` extends the prefix.
  auto select = [&](bool by_mass, uint32_t floor_key, uint64_t need, uint64_t& total) -> uint32_t {
    uint32_t prefix = 0, pmask = 0;
    uint64_t above = 0;
    const int shifts[3] = {21, 10, 0}, widths[3] = {11, 11, 10};
    total = 0;
    for (int lvl = 0; lvl < 3; ++lvl) {
      const int sh = shifts[lvl], nb = 1 << widths[lvl];
      for (int i = threadIdx.x; i < kBins; i += kThreads) s_hist[i] = 0;
      __syncthreads();
      row.each([&](int, float x) {
        const uint32_t k = fkey(x);
        if (k >= floor_key && (k & pmask) == prefix)
          atomicAdd((unsigned long long*)&s_hist[(k >> sh) & (nb - 1)], by_mass ? (unsigned long long)fmass(x, mx) : 1ull);
      });
      __syncthreads();
      if (threadIdx.x < 64) {
        // lane l owns bins [l * nb / 64, (l + 1) * nb / 64); suffix sums from the top bin down
        const int per = nb / 64, lo = threadIdx.x * per;
        uint64_t mine = 0;
        for (int i = 0; i < per; ++i) mine += s_hist[lo + i];
        if (lvl == 0) total = wave_sum_u64(mine);  // (uniform: everything at or above floor_key)
        // inclusive suffix scan of lane sums across the wave (from lane 63 down)
        uint64_t suf = mine;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const uint64_t v = __shfl_down(suf, o, kWave);
          if ((int)threadIdx.x + o < 64) suf += v;
        }
        // the lane whose range holds the crossing: above + suffix(l) >= need > above + suffix(l + 1)
        const uint64_t next = __shfl_down(suf, 1, kWave);
        const uint64_t suf_next = threadIdx.x < 63 ? next : 0;
        if (above + suf >= need && above + suf_next < need) {
          uint64_t run = above + suf_next;
          int d = lo + per - 1;
          for (; d > lo; --d) {
            if (run + s_hist[d] >= need) break;
            run += s_hist[d];
          }
          s_sel[0] = (uint32_t)d;
          s_sel[1] = (uint32_t)(run & 0xffffffffu);
          s_sel[2] = (uint32_t)(run >> 32);
        }
        if (lvl == 0) s_red[0] = total;
      }
      __syncthreads();
      const uint32_t d = s_sel[0];
      above = (uint64_t)s_sel[1] | ((uint64_t)s_sel[2] << 32);
      total = s_red[0];
      prefix |= d << sh;
      pmask |= (uint32_t)(nb - 1) << sh;
      __syncthreads();
    }
    return prefix;
  };

  // ---- top-k threshold (key of the k-th largest logit; ties kept)
  const int k = top_k ? top_k[b] : top_k_all;
  uint64_t dummy;
  if (!have_k && k > 0 && k < vocab) thr = select(false, 0u, (uint64_t)k, dummy);

  // ---- top-p threshold over the top-k set
  const float pp = top_p ? top_p[b] : top_p_all;
  if (pp < 1.f && !have_p) {
    // mass of the top-k set first (the first level's histogram total), then the selection; a row handed
    // back for its ties: their number too, since the threshold stands where the mass above it does not
    // reach the target (5 % of a top-k row's time, so only there)
    uint64_t mk = 0, ties = 0;
    if (have_k) {
      row.each([&](int, float x) {
        const uint32_t key = fkey(x);
        if (key >= thr) mk += fmass(x, mx);
        ties += key == thr;
      });
      ties = block_sum_u64(ties, s_red) * fmass(key_float(thr), mx);
    } else {
      row.each([&](int, float x) { if (fkey(x) >= thr) mk += fmass(x, mx); });
    }
    mk = block_sum_u64(mk, s_red);
    double needd = ceil((double)fmaxf(pp, 0.f) * (double)mk);
    uint64_t need = needd < 1.0 ? 1 : (uint64_t)needd;
    if (need > mk) need = mk;
    if (mk > 0 && need + ties <= mk) {
      uint64_t tot;
      const uint32_t tp = select(true, thr, need, tot);
      thr = tp > thr ? tp : thr;
    }
  }

  // ---- sample: kept mass per tile, the tile holding the target, then the thread and token
  if (!have_tiles) {
    for (int t = threadIdx.x; t < ntiles; t += kThreads) s_tile[t] = 0;
    __syncthreads();
    constexpr int E = RowT::E;
    uint64_t m = 0;
    int cur = 0;
    row.each([&](int i, float x) {
      const int t = i / (kThreads * E);
      if (t != cur) {  // (tiles come in increasing order)
        if (m) atomicAdd((unsigned long long*)&s_tile[cur], (unsigned long long)m);
        m = 0;
        cur = t;
      }
      if (fkey(x) >= thr) m += fmass(x, mx);
    });
    if (m) atomicAdd((unsigned long long*)&s_tile[cur], (unsigned long long)m);
  }
  __syncthreads();
  uint64_t ms = 0;
  for (int t = 0; t < ntiles; ++t) ms += s_tile[t];  // (every thread: uniform)
  int32_t token = -1;
  if (ms > 0) {
    const double uu = fminf(fmaxf(uniform[b], 0.f), 1.f);
    uint64_t target = (uint64_t)(uu * (double)ms);
    if (target >= ms) target = ms - 1;
    int tt = 0;
    uint64_t before = 0;
    while (tt < ntiles - 1 && before + s_tile[tt] <= target) before += s_tile[tt++];
    // inside tile tt: each thread's kept mass, exclusive scan, then the owner walks its logits
    uint64_t mine = 0;
    row.tile(tt, [&](int, float x) { if (fkey(x) >= thr) mine += fmass(x, mx); });
    // block exclusive scan: inclusive within each wave, then the waves' totals
    uint64_t inc = mine;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint64_t v = __shfl_up(inc, o, kWave);
      if (lane >= o) inc += v;
    }
    if (lane == 63) s_scan[wv] = inc;
    __syncthreads();
    uint64_t off = before;
    for (int i = 0; i < wv; ++i) off += s_scan[i];
    const uint64_t start = off + inc - mine;
    if (mine > 0 && start <= target && target < start + mine) {
      uint64_t run = start;
      int found = -1;
      row.tile(tt, [&](int i, float x) {
        if (found < 0 && fkey(x) >= thr) {
          run += fmass(x, mx);
          if (run > target) found = i;
        }
      });
      out[b] = found;
    }
  } else if (threadIdx.x == 0) {
    out[b] = token;  // (no token carries mass: an all-NaN or empty row)
  }
}

// Which kernels sample a row: its whole distribution (no top-k, no top-p filter), a top-k filter with
// k <= kTopKMax (then any top-p), a top-p filter alone, or anything else (the one-workgroup kernel).
enum RowKind : int { kWholeRow = 0, kTopKRow = 1, kTopPRow = 2, kOtherRow = 3 };
constexpr int kTopKMax = 256;
__host__ __device__ __forceinline__ int row_kind_of(int k, float pp, int vocab) {
  if (k <= 0 || k >= vocab) return pp < 1.f ? kTopPRow : kWholeRow;
  return k <= kTopKMax ? kTopKRow : kOtherRow;
}
__device__ __forceinline__ int row_kind(int b, int vocab, const int32_t* top_k, int32_t top_k_all,
                                        const float* top_p, float top_p_all) {
  return row_kind_of(top_k ? top_k[b] : top_k_all, top_p ? top_p[b] : top_p_all, vocab);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void sample_kernel(const T* logits, int64_t row_stride, int vocab,
                                                          const int32_t* top_k, int32_t top_k_all,
                                                          const float* top_p, float top_p_all,
                                                          const float* uniform, int32_t* out, int split,
                                                          const int32_t* fallback, const ToppBin* known) {
  __shared__ SampleLds L;
  const int b = blockIdx.x;
  // with the split kernels in use, all kinds but kOtherRow are theirs, except the rows they handed
  // back (fallback[b])
  const int how = split ? fallback[b] : (int)kNotBack;
  if (split && row_kind(b, vocab, top_k, top_k_all, top_p, top_p_all) != kOtherRow && how == kNotBack) return;
  const T* p = logits + (int64_t)b * row_stride;
  const Row<T> row{p, vocab, ((uintptr_t)p % 16) == 0};
  sample_row<T>(row, L, b, vocab, top_k, top_k_all, top_p, top_p_all, uniform, out, how, known + b);
}

// ---- Rows over many workgroups.  One workgroup per row leaves half the chip idle and is bound by the
// vector ALU of the CUs it has (eight passes over a top-p row: 165 us for 32 rows of 151,936), so rows
// are cut into slices of kSliceTiles tiles of kSplitTile logits, one workgroup per (slice, row), in
// launches that every kind of row shares:
//   split_scan_kernel    the logits scaled, if asked for; each slice's largest and smallest logit, and
//                        the largest of each group of logits (256 of them at a vocabulary of 151,936)
//   split_pass_kernel    whole rows: each tile's mass, then the workgroup that finishes the row's last
//                        slice finds the tile and the token; top-k rows: the token; top-p rows: the
//                        mass by distance from the row's largest logit
//   split_finish_kernel  top-p rows: the threshold and the token
//   sample_kernel        other rows, and rows handed back, with what is known of them (Back)
// All masses and targets are the integers sample_row computes, so the token is identical.
// What bounds them: the scan moves the logits, the penalties and the scaled logits (156 MB in 33 us at
// 128 x 151,936 fp16); the later launches are chains of latencies (arrivals, LDS rounds) beside 3 to 4
// TB/s of reading.  128 rows of 151,936 fp16 logits, penalty and temperature, two requests in eight
// top-p alone and five top-k: 260 us when every filtered row but small top-k ran on one workgroup and
// the scaling was a launch of its own, 96 us; without the scaling 223 and 75; all top_k 50 / top_p 0.9:
// 54.8 and 32.5; one row: 34.7 and 22.4.
constexpr int kSplitThreads = 256;
constexpr int kSplitTile = kSplitThreads * 8;  // 8 logits per thread
constexpr int kSliceTiles = 8;
constexpr int kMaxSplitTiles = 2048;           // vocabularies up to 4 M

constexpr int kCandCap = 512;    // candidates a slice hands over for a top-p row

constexpr int kGroups = 1024;    // group maxima per row at most
constexpr int kPCandMax = 2048;  // candidates of a top-p row (at 512 bins and 1024 of them, a wide body at a high
                                 // temperature went over, and the one row handed back took 45 us)

__host__ __device__ inline int split_tiles(int vocab) { return (vocab + kSplitTile - 1) / kSplitTile; }
__host__ __device__ inline int split_slices(int vocab) { return (split_tiles(vocab) + kSliceTiles - 1) / kSliceTiles; }
// The groups whose maxima a row keeps, at most kGroups of them and as small as that allows: a thread's
// logits of 2^tg tiles of a slice, over 2^gl neighbouring threads.
struct GroupShape {
  int tg, gl, per_slice, ps, n;  // (per_slice = 2^ps)
};
inline GroupShape group_shape(int vocab) {
  const int S = split_slices(vocab);
  GroupShape g{0, 0, 0, 0, 0};
  auto count = [&]() { return S * ((kSliceTiles * kSplitThreads) >> (g.tg + g.gl)); };
  while (count() > kGroups && (1 << g.tg) < kSliceTiles) ++g.tg;
  while (count() > kGroups && g.gl < 6) ++g.gl;
  g.per_slice = (kSliceTiles * kSplitThreads) >> (g.tg + g.gl);
  while ((1 << g.ps) < g.per_slice) ++g.ps;
  g.n = S * g.per_slice;
  return g;
}

constexpr int kCountStride = 32;
static_assert(kCandCap <= kPBins, "candidates in the bins' place");
struct SplitWs {
  uint64_t* tmass;    // [rows][ntiles] tile masses (whole and top-p rows)
  uint64_t* hist;     // [rows][slices][kPBins] masses by bin (top-p rows, split_pass_kernel)
  uint64_t* cand;     // the same area: kCandCap candidates a slice, index << 32 | key (split_finish_kernel)
  ToppBin* bin;       // [rows] where the threshold lies (top-p rows; top-k rows that are handed back)
  uint16_t* gmax;     // [rows][kGroups] group maxima: the keys' upper halves
  float* smax;        // [rows][slices] slice maxima
  float* smin;        // [rows][slices] slice minima
  int32_t* ncand;     // [rows][slices] candidates per slice, -1: more than kCandCap
  int32_t* counter;   // [rows][kCountStride] slices finished: a cache line each
  int32_t* fallback;  // [rows] whether handed back to the one-workgroup kernel (Back)
  GroupShape g;
};
__host__ __device__ inline int64_t split_ws_bytes(int rows, int vocab) {
  const int64_t S = split_slices(vocab);
  return (int64_t)rows * (split_tiles(vocab) * 8 + S * kPBins * 8 + (int64_t)sizeof(ToppBin) + kGroups * 2 + S * 12 + kCountStride * 4 + 4);
}
inline SplitWs split_ws(void* ws, int rows, int vocab) {
  const int64_t S = split_slices(vocab);
  char* c = reinterpret_cast<char*>(ws);
  auto take = [&](int64_t bytes) {
    char* p = c;
    c += (int64_t)rows * bytes;
    return p;
  };
  SplitWs w;
  w.tmass = reinterpret_cast<uint64_t*>(take(split_tiles(vocab) * 8));
  w.hist = reinterpret_cast<uint64_t*>(take(S * kPBins * 8));
  w.cand = w.hist;
  w.bin = reinterpret_cast<ToppBin*>(take(sizeof(ToppBin)));
  w.gmax = reinterpret_cast<uint16_t*>(take(kGroups * 2));
  w.smax = reinterpret_cast<float*>(take(S * 4));
  w.smin = reinterpret_cast<float*>(take(S * 4));
  w.ncand = reinterpret_cast<int32_t*>(take(S * 4));
  w.counter = reinterpret_cast<int32_t*>(take(kCountStride * 4));
  w.fallback = reinterpret_cast<int32_t*>(take(4));
  w.g = group_shape(vocab);
  return w;
}
static_assert(kMaxSplitTiles / kSliceTiles * (kSplitThreads >> 6) <= kGroups, "the largest rows' groups");

// Thread t's 8 logits of tile j: indices j * kSplitTile + 8 t .. + 7 (ok: inside the row).
template <typename T>
__device__ __forceinline__ void load8(const T* p, int vocab, bool vec, int j, float (&x)[8], bool (&ok)[8]) {
  const int base = j * kSplitTile + 8 * (int)threadIdx.x;
  if (vec && base + 8 <= vocab) {
    T e[8];
#pragma unroll
    for (int v = 0; v < (int)(8 * sizeof(T) / 16); ++v) {
      const uint4 w = *reinterpret_cast<const uint4*>(p + base + v * (16 / sizeof(T)));
      __builtin_memcpy(e + v * (16 / sizeof(T)), &w, 16);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      x[k] = to_f32(e[k]);
      ok[k] = true;
    }
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      ok[k] = base + k < vocab;
      x[k] = ok[k] ? to_f32(p[base + k]) : 0.f;
    }
  }
}

// A slice's tiles for thread t, all loads issued before any is used: 16-byte vectors from
// clamped in-bounds addresses (a load under a divergent branch would be waited for at the
// branch's end, one tile at a time); get() then reads them, or the row with element loads
// where a vector would cross its end (or the row is not 16-byte aligned).
template <typename T>
struct SliceLoad {
  static constexpr int R = 8 * sizeof(T) / 16;  // vectors per thread per tile
  uint4 raw[kSliceTiles][R];
  __device__ __forceinline__ void issue(const T* p, int vocab, bool vec, int j0, int j1) {
    if (!(vec && vocab >= 8)) return;  // (uniform)
    const int last = (vocab - 8) / 8 * 8;
#pragma unroll
    for (int jj = 0; jj < kSliceTiles; ++jj) {
      const int j = min(j0 + jj, j1 - 1);
      const int base = min(j * kSplitTile + 8 * (int)threadIdx.x, last);
#pragma unroll
      for (int v = 0; v < R; ++v) raw[jj][v] = *reinterpret_cast<const uint4*>(p + base + v * (16 / sizeof(T)));
    }
  }
  __device__ __forceinline__ void get_raw(const T* p, int vocab, bool vec, int j, int jj, T (&e)[8],
                                          bool (&ok)[8]) const {
    const int base = j * kSplitTile + 8 * (int)threadIdx.x;
    if (vec && vocab >= 8 && base + 8 <= vocab) {
      __builtin_memcpy(e, raw[jj], 8 * sizeof(T));
#pragma unroll
      for (int k = 0; k < 8; ++k) ok[k] = true;
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        ok[k] = base + k < vocab;
        if (ok[k]) e[k] = p[base + k];
      }
    }
  }
  __device__ __forceinline__ void get(const T* p, int vocab, bool vec, int j, int jj, float (&x)[8],
                                      bool (&ok)[8]) const {
    T e[8];
    get_raw(p, vocab, vec, j, jj, e, ok);
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = ok[k] ? to_f32(e[k]) : 0.f;
  }
};

// The tiles' sums of a slice, each over the workgroup: add() per tile, then store() by all threads.
struct TileSums {
  uint64_t (*red)[4];  // [kSliceTiles][4] in LDS
  __device__ __forceinline__ void add(int jj, uint64_t m) const {
    m = wave_sum_u64(m);
    if ((threadIdx.x & 63) == 0) red[jj][threadIdx.x >> 6] = m;
  }
  // (a row of one slice: for the workgroup itself)
  __device__ __forceinline__ void keep(uint64_t* s_tile, int n) const {
    __syncthreads();
    const int t = threadIdx.x;
    if (t < n) s_tile[t] = red[t][0] + red[t][1] + red[t][2] + red[t][3];
  }
  // (written through to device scope)
  __device__ __forceinline__ void store(uint64_t* tm, int n) const {
    __syncthreads();
    const int t = threadIdx.x;
    if (t < n)
      __hip_atomic_store(tm + t, red[t][0] + red[t][1] + red[t][2] + red[t][3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};
// Largest of mx over the workgroup; red: 4 floats.
__device__ __forceinline__ float block_max256(float mx, float* red) {
  mx = wave_max_f32(mx);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}
// Largest of mx (x) and smallest of mn (y) over the workgroup; red: 8 floats.
__device__ __forceinline__ float2 block_range256(float mx, float mn, float* red) {
  mx = wave_max_f32(mx);
  mn = wave_max_f32(-mn);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6] = mx;
    red[4 + (threadIdx.x >> 6)] = mn;
  }
  __syncthreads();
  return make_float2(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])),
                     -fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7])));
}
// One scaled logit: x / penalty rounded to T, then / temperature in fp32, both IEEE divisions (a divisor
// of 1 leaves the value unchanged).
template <typename T>
__device__ __forceinline__ float scale_logit(T xv, T pv, bool pen, float t) {
  float y = to_f32(xv);
  if (pen) {
    const float d = to_f32(pv);
    if (d != 1.f) y = to_f32(from_f32<T>(y / d));
  }
  if (t != 1.f) y = y / t;
  return y;
}

// What split_scan_kernel<T, true> scales by, and where the fp32 results go (rows of out_stride floats,
// a multiple of 4).
template <typename T>
struct ScaleArgs {
  const T* penalty;
  int64_t penalty_stride;
  int32_t slots;
  const int32_t* rows;
  const float* temperature;
  float* out;
  int64_t out_stride;
};

// WHOLE, here and in the pass: the host knows that every row is a whole row, and the kernels hold nothing
// else (one row of 1000 logits 10.5 -> 9.0 us, 128 of 32,000 16.8 -> 15.2, of 151,936 33.7 -> 30.4, in a graph,
// with rows of one slice done without an arrival and the token's tile found without a barrier; 9.2, 15.1 and
// 32.0 when the kinds had launches of their own).
template <typename T, bool SCALE, bool WHOLE>
__global__ __launch_bounds__(kSplitThreads) void split_scan_kernel(const T* logits, int64_t row_stride, int vocab,
                                                                   const int32_t* top_k, int32_t top_k_all,
                                                                   const float* top_p, float top_p_all,
                                                                   ScaleArgs<T> sc, SplitWs ws) {
  __shared__ float red[8];
  const int s = blockIdx.x, b = blockIdx.y, S = gridDim.x, ntiles = split_tiles(vocab);
  if (s == 0 && threadIdx.x == 0) {  // (read by the later launches on this stream)
    ws.counter[b * kCountStride] = 0;
    ws.fallback[b] = 0;
  }
  const int kind = WHOLE ? (int)kWholeRow : row_kind(b, vocab, top_k, top_k_all, top_p, top_p_all);
  if (!SCALE && kind == kOtherRow) return;
  const T* p = logits + (int64_t)b * row_stride;
  const bool vec = ((uintptr_t)p % 16) == 0;
  const int j0 = s * kSliceTiles, j1 = min(j0 + kSliceTiles, ntiles);
  const GroupShape& g = ws.g;
  uint16_t* gm = ws.gmax + (int64_t)b * kGroups + s * g.per_slice;
  float mn = INFINITY, mx = -INFINITY, gx = -INFINITY;  // the slice's smallest and largest, the group's largest so far
  auto see = [&](const float (&x)[8], const bool (&ok)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      gx = ok[k] ? fmaxf(gx, x[k]) : gx;
      if constexpr (!WHOLE) mn = ok[k] ? fminf(mn, x[k]) : mn;
    }
  };
  auto group_end = [&](int jj) __attribute__((always_inline)) {
    if ((kind == kTopKRow || kind == kTopPRow) && ((jj + 1) & ((1 << g.tg) - 1)) == 0) {  // (uniform)
      mx = fmaxf(mx, gx);
      for (int o = 1; o < (1 << g.gl); o <<= 1) gx = fmaxf(gx, __shfl_xor(gx, o, kWave));
      const int at = ((jj >> g.tg) * kSplitThreads + (int)threadIdx.x) >> g.gl;
      if ((threadIdx.x & ((1 << g.gl) - 1)) == 0) gm[at] = (uint16_t)(fkey(gx) >> 16);  // (no number in it: as -inf)
      gx = -INFINITY;
    }
  };
  if constexpr (!SCALE) {
    SliceLoad<T> sl;
    sl.issue(p, vocab, vec, j0, j1);
#pragma unroll
    for (int jj = 0; jj < kSliceTiles; ++jj) {
      if (j0 + jj < j1) {
        float x[8];
        bool ok[8];
        sl.get(p, vocab, vec, j0 + jj, jj, x, ok);
        see(x, ok);
      }
      group_end(jj);
    }
  } else {
    // a tile at a time, the next one's vectors on their way: the divisions are long, and eight tiles
    // unrolled with their logits and penalties in registers spilled (128 x 151,936 fp16: 50 us; four at
    // once 38, two ahead 36, one ahead 32)
    constexpr int R = 8 * sizeof(T) / 16;
    float* o = sc.out + (int64_t)b * sc.out_stride;
    const float temp = sc.temperature ? sc.temperature[b] : 1.f;
    const int pr = sc.penalty ? sc.rows[b] : 0;
    const bool bad = sc.penalty && (pr < 0 || pr >= sc.slots);  // no such penalty row: the row reads as NaN
    const T* pen = sc.penalty ? sc.penalty + (int64_t)(bad ? 0 : pr) * sc.penalty_stride : p;
    const bool has_pen = sc.penalty != nullptr, whole = vec && ((uintptr_t)pen % 16) == 0 && vocab >= 8;
    const int last = (vocab - 8) / 8 * 8;
    uint4 nx[R], np[R];
    auto issue = [&](int j) __attribute__((always_inline)) {  // (clamped: whole vectors inside the row)
      const int base = min(j * kSplitTile + 8 * (int)threadIdx.x, last);
#pragma unroll
      for (int v = 0; v < R; ++v) {
        nx[v] = *reinterpret_cast<const uint4*>(p + base + v * (16 / sizeof(T)));
        np[v] = *reinterpret_cast<const uint4*>(pen + base + v * (16 / sizeof(T)));
      }
    };
    if (whole) issue(j0);
#pragma unroll 1
    for (int jj = 0; jj < kSliceTiles; ++jj) {
      if (j0 + jj < j1) {
        const int base = (j0 + jj) * kSplitTile + 8 * (int)threadIdx.x;
        T xs[8], ps[8];
        bool ok[8];
        if (whole) {
          __builtin_memcpy(xs, nx, 8 * sizeof(T));
          __builtin_memcpy(ps, np, 8 * sizeof(T));
          issue(min(j0 + jj + 1, j1 - 1));
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          ok[k] = base + k < vocab;
          if (ok[k] && !(whole && base + 8 <= vocab)) {
            xs[k] = p[base + k];
            ps[k] = pen[base + k];
          }
        }
        float x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = bad ? __builtin_nanf("") : scale_logit<T>(xs[k], ps[k], has_pen, temp);
        if (base + 8 <= vocab) {
          *reinterpret_cast<float4*>(o + base) = make_float4(x[0], x[1], x[2], x[3]);
          *reinterpret_cast<float4*>(o + base + 4) = make_float4(x[4], x[5], x[6], x[7]);
        } else {
#pragma unroll
          for (int k = 0; k < 8; ++k)
            if (ok[k]) o[base + k] = x[k];
        }
        see(x, ok);
      }
      group_end(jj);
    }
  }
  if constexpr (WHOLE) {
    const float r = block_max256(gx, red);
    if (threadIdx.x == 0) ws.smax[(int64_t)b * S + s] = r;
  } else if (kind == kWholeRow || kind == kTopPRow) {
    const float2 r = block_range256(fmaxf(mx, gx), mn, red);
    if (threadIdx.x == 0) {
      ws.smax[(int64_t)b * S + s] = r.x;
      ws.smin[(int64_t)b * S + s] = r.y;
    }
  }
}

// Inclusive sum over the threads below and at this one (and, in `all`, over all of them).
__device__ __forceinline__ uint64_t block_scan256(uint64_t v, uint64_t* red, uint64_t& all) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t y = __shfl_up(v, o, kWave);
    if (lane >= o) v += y;
  }
  __syncthreads();
  if (lane == 63) red[wv] = v;
  __syncthreads();
  for (int i = 0; i < wv; ++i) v += red[i];
  all = red[0] + red[1] + red[2] + red[3];
  return v;
}

// Each of n <= 256 entries against every one, by the workgroup: 256 / n (a power of two) neighbouring
// threads share an entry and call f(i) for their part of i = 0 .. n - 1; entry() is the thread's.
struct Pairs {
  int n, shift;
  __device__ __forceinline__ Pairs(int n_) : n(n_), shift(n_ <= 32 ? 3 : n_ <= 64 ? 2 : n_ <= 128 ? 1 : 0) {}
  __device__ __forceinline__ int entry() const { return (int)threadIdx.x >> shift; }
  __device__ __forceinline__ bool first() const { return (threadIdx.x & ((1 << shift) - 1)) == 0; }
  // The mass of the entries with key >= lo and index < lim.  The entries are read four at a time before
  // any is used: one by one, each LDS read's latency is waited out.
  __device__ __forceinline__ uint64_t mass(const uint64_t* cand, const uint64_t* mass, uint32_t lo, uint32_t lim) const {
    const int parts = 1 << shift, sub = threadIdx.x & (parts - 1);
    uint64_t f = 0;
#pragma unroll 1
    for (int i0 = sub; i0 < n; i0 += 4 * parts) {
      uint64_t c[4], m[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int i = min(i0 + x * parts, n - 1);
        c[x] = cand[i];
        m[x] = mass[i];
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int x = 0; x < 4; ++x)
        f += i0 + x * parts < n && (uint32_t)c[x] >= lo && (uint32_t)(c[x] >> 32) < lim ? m[x] : 0;
    }
#pragma unroll 1
    for (int o = 1; o < parts; o <<= 1) f += __shfl_xor(f, o, kWave);
    return f;
  }
};
// A wave's largest (sum) into LDS.  Reduced in registers first: from an atomic whose lanes hold different
// values for one address the compiler makes a loop over the lanes, about 1 us.
__device__ __forceinline__ void wave_to_lds_max(uint32_t* p, uint32_t v) {
  v = wave_max_u32(v);
  if ((threadIdx.x & 63) == 0) atomicMax(p, v);
}
__device__ __forceinline__ void wave_to_lds_sum(uint64_t* p, uint64_t v) {
  v = wave_sum_u64(v);
  if ((threadIdx.x & 63) == 0) atomicAdd((unsigned long long*)p, (unsigned long long)v);
}
// The token of a whole or top-p row from its tiles' kept masses (in s_tile, for every thread): the
// tile holding the target, then each thread's kept mass in it, an exclusive scan in thread (=
// vocabulary) order, and the owner walks its 8 logits.  Kept: key >= thr.  redu: written here, read by
// nobody since the last barrier.
template <typename T>
__device__ __forceinline__ void pick_token(const T* p, int vocab, bool vec, float mx, uint32_t thr, const uint64_t* s_tile,
                                           int ntiles, float u, int32_t* out, uint64_t* redu) {
  // lane l: the tiles [per l, per (l + 1)); every wave for itself, without a barrier
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int per = (ntiles + kWave - 1) / kWave, q0 = per * lane;
  uint64_t own = 0;
  for (int j = q0; j < min(q0 + per, ntiles); ++j) own += s_tile[j];
  uint64_t upto = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t v = __shfl_up(upto, o, kWave);
    if (lane >= o) upto += v;
  }
  const uint64_t ms = __shfl(upto, 63, kWave);
  if (ms == 0) {  // (uniform)
    if (threadIdx.x == 0) *out = -1;  // (no token carries mass: an all-NaN row)
    return;
  }
  const double uu = fminf(fmaxf(u, 0.f), 1.f);
  uint64_t target = (uint64_t)(uu * (double)ms);
  if (target >= ms) target = ms - 1;
  const int at = __builtin_ctzll(__ballot(upto > target));  // the lane whose tiles hold it
  uint64_t before = __shfl(upto - own, at, kWave);
  int tt = per * at;
  while (before + s_tile[tt] <= target) before += s_tile[tt++];
  float x[8];
  bool ok[8];
  load8(p, vocab, vec, tt, x, ok);
  uint64_t mine = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    ok[k] = ok[k] && fkey(x[k]) >= thr;
    if (ok[k]) mine += fmass(x[k], mx);
  }
  uint64_t inc = mine;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t v = __shfl_up(inc, o, kWave);
    if (lane >= o) inc += v;
  }
  if (lane == 63) redu[wv] = inc;
  __syncthreads();
  uint64_t off = before;
  for (int i = 0; i < wv; ++i) off += redu[i];
  const uint64_t start = off + inc - mine;
  if (mine > 0 && start <= target && target < start + mine) {
    uint64_t run = start;
    int found = -1;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (found < 0 && ok[k]) {
        run += fmass(x[k], mx);
        if (run > target) found = tt * kSplitTile + 8 * (int)threadIdx.x + k;
      }
    }
    *out = found;
  }
}
// Arrival of a slice whose results are written through to device scope: true in the workgroup that
// finishes the row's last slice.
__device__ __forceinline__ bool slice_arrive(int32_t* counter, int S, int* s_last) {
  __builtin_amdgcn_s_waitcnt(0x0F70);  // this thread's results are complete (device-visible)
  __syncthreads();
  if (threadIdx.x == 0) *s_last = atomicAdd(counter, 1) == S - 1;
  __syncthreads();
  return *s_last;
}
__device__ __forceinline__ void st_dev_u64(uint64_t* p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename V>
__device__ __forceinline__ V ld_dev(const V* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A row's largest and smallest logit from its slices' (written by the scan's launch).
__device__ __forceinline__ float2 row_range(const SplitWs& ws, int b, int S, float* red) {
  float mx = -INFINITY, mn = INFINITY;
  for (int i = threadIdx.x; i < S; i += kSplitThreads) {
    mx = fmaxf(mx, ws.smax[(int64_t)b * S + i]);
    mn = fminf(mn, ws.smin[(int64_t)b * S + i]);
  }
  return block_range256(mx, mn, red);
}

template <typename T>
__device__ __forceinline__ void whole_slice(const T* p, int vocab, bool vec, const SliceLoad<T>& sl, int s, int b, int S,
                                            const float* uniform, int32_t* out, const SplitWs& ws, uint64_t* s_tile,
                                            float* redf, uint64_t (*redu)[4], int* s_last) {
  const TileSums sums{redu};
  const int ntiles = split_tiles(vocab), j0 = s * kSliceTiles, j1 = min(j0 + kSliceTiles, ntiles);
  float mx = -INFINITY;
  for (int i = threadIdx.x; i < S; i += kSplitThreads) mx = fmaxf(mx, ws.smax[(int64_t)b * S + i]);
  mx = block_max256(mx, redf);
  // this slice's tile masses, written through to device scope
  uint64_t* tm = ws.tmass + (int64_t)b * ntiles;
#pragma unroll
  for (int jj = 0; jj < kSliceTiles; ++jj) {
    if (j0 + jj >= j1) break;  // (uniform)
    float x[8];
    bool ok[8];
    sl.get(p, vocab, vec, j0 + jj, jj, x, ok);
    uint64_t m = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (ok[k]) m += fmass(x[k], mx);
    sums.add(jj, m);
  }
  if (S == 1) {  // (uniform)
    sums.keep(s_tile, ntiles);
  } else {
    sums.store(tm + j0, j1 - j0);
    if (!slice_arrive(&ws.counter[b * kCountStride], S, s_last)) return;
    for (int j = threadIdx.x; j < ntiles; j += kSplitThreads) s_tile[j] = ld_dev(tm + j);
  }
  __syncthreads();
  pick_token(p, vocab, vec, mx, 0u, s_tile, ntiles, uniform[b], out + b, redu[0]);
}

// ---- Top-p rows.  The row's masses are binned by distance from its largest logit (kPBins bins over
// the range that carries mass: a monotone function of the logit, so the bins are in the logits'
// order); the bin where the mass from the top reaches the target holds the threshold, and the workgroup
// that finishes the row's last slice finds it.  In the next launch logits in the bins above are kept,
// those in it are candidates (a few hundred of 151,936), and the last slice's workgroup selects the
// exact threshold among them.  That launch reads only the groups whose largest logit reaches the bin.
template <typename T>
__device__ __forceinline__ void topp_hist(const T* p, int vocab, bool vec, const SliceLoad<T>& sl, int s, int b, int S,
                                          float pp, int32_t* out, const SplitWs& ws, uint64_t* s_hist, float* redf,
                                          uint64_t* redu, int* s_last) {
  const int ntiles = split_tiles(vocab), j0 = s * kSliceTiles, j1 = min(j0 + kSliceTiles, ntiles), t = threadIdx.x;
  for (int i = t; i < kPBins; i += kSplitThreads) s_hist[i] = 0;
  const PBins bins(row_range(ws, b, S, redf));  // (synchronises)
#pragma unroll
  for (int jj = 0; jj < kSliceTiles; ++jj) {
    if (j0 + jj >= j1) break;  // (uniform)
    float x[8];
    bool ok[8];
    sl.get(p, vocab, vec, j0 + jj, jj, x, ok);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint64_t m = ok[k] ? fmass(x[k], bins.mx) : 0;
      if (m) atomicAdd((unsigned long long*)&s_hist[bins.of(x[k])], (unsigned long long)m);
    }
  }
  __syncthreads();
  uint64_t* h = ws.hist + (int64_t)b * S * kPBins;
  for (int i = t; i < kPBins; i += kSplitThreads) st_dev_u64(h + (int64_t)s * kPBins + i, s_hist[i]);
  if (!slice_arrive(&ws.counter[b * kCountStride], S, s_last)) return;
  // ---- the bin that holds the threshold; thread t: bins 4t .. 4t + 3
  static_assert(kPBins == 4 * kSplitThreads, "four bins a thread");
  uint64_t hb[4] = {0, 0, 0, 0};
#pragma unroll 4
  for (int i = 0; i < S; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) hb[e] += ld_dev(h + (int64_t)i * kPBins + 4 * t + e);
  const uint64_t own = hb[0] + hb[1] + hb[2] + hb[3];
  uint64_t mk;
  const uint64_t incl = block_scan256(own, redu, mk), excl = incl - own;
  const double needd = ceil((double)fmaxf(pp, 0.f) * (double)mk);
  uint64_t need = needd < 1.0 ? 1 : (uint64_t)needd;
  if (need > mk) need = mk;
  if (t == 0) ws.counter[b * kCountStride] = 0;  // (for the next launch's arrivals)
  if (mk == 0) {  // (no token carries mass)
    if (t == 0) {
      ws.bin[b].bin = -1;
      out[b] = -1;
    }
  } else if (incl >= need && excl < need) {
    uint64_t above = excl;
    int e = 0;
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const bool on = e == x && above + hb[x] < need;
      above += on ? hb[x] : 0;
      e += on ? 1 : 0;
    }
    ws.bin[b] = ToppBin{above, need, bins.mx, bins.scale, 4 * t + e};
    // at least this many logits carry the bin's mass; too many for the next launch, which then leaves the
    // row alone (ties, mostly)
    uint64_t mine = 0;
#pragma unroll
    for (int x = 0; x < 4; ++x) mine = e == x ? hb[x] : mine;
    const float most = __expf(-(float)(4 * t + e) / bins.scale) * 4294967296.0f;  // (of one of them)
    // (several slices do not share them evenly)
    const int room = min(kPCandMax, S == 1 ? kCandCap : S * (kCandCap - kCandCap / 8));
    if ((float)mine > (float)room * (1.01f * most + 1.f)) ws.fallback[b] = kBackBin;
  }
}

struct ToppLds {
  uint64_t cand[kPCandMax];
  uint64_t mass[kSplitThreads];  // (of up to 256 candidates)
  uint64_t hist[kSplitThreads];
  uint64_t redu[4], tsum[kSliceTiles][4];
  uint64_t above;
  int off[kMaxSplitTiles / kSliceTiles + 1];
  uint32_t diff, thr;
  int bin, n, last;
};

template <typename T>
__device__ __forceinline__ void topp_finish(const T* p, int vocab, int s, int b, int S, const float* uniform, int32_t* out,
                                            const SplitWs& ws, ToppLds& L, uint64_t* s_tile) {
  const int t = threadIdx.x;
  const int ntiles = split_tiles(vocab), j0 = s * kSliceTiles, j1 = min(j0 + kSliceTiles, ntiles);
  const bool vec = ((uintptr_t)p % 16) == 0;
  const GroupShape& g = ws.g;
  const uint16_t* gm = ws.gmax + (int64_t)b * kGroups + s * g.per_slice;
  const ToppBin tb = ws.bin[b];
  const int cb = (int)tb.bin;
  const uint64_t above = tb.above, need = tb.need;
  if (cb < 0 || ws.fallback[b] != kNotBack) return;  // (uniform; the token is written, or the row handed back)
  if (t == 0) L.n = 0, L.diff = 0;
  const PBins bins(tb.mx, tb.scale);
  __syncthreads();
  // ---- this slice: its tiles' mass above the bin, and its candidates, written through to device scope
  const TileSums sums{L.tsum};
  uint64_t* tm = ws.tmass + (int64_t)b * ntiles;
  uint64_t* pc = ws.cand + ((int64_t)b * S + s) * kPBins;
  // a group's largest logit is at most the float of its key's upper half and all lower bits set; threads
  // of groups that do not reach the bin load the row's first vector instead
  constexpr int R = 8 * sizeof(T) / 16;
  const bool vecs = vec && vocab >= 8;
  bool act[kSliceTiles];
  uint4 raw[kSliceTiles][R];
  {
    uint32_t gk[kSliceTiles];
#pragma unroll
    for (int jj = 0; jj < kSliceTiles; ++jj) gk[jj] = gm[((jj >> g.tg) * kSplitThreads + t) >> g.gl];
#pragma unroll
    for (int jj = 0; jj < kSliceTiles; ++jj) {
      const int base = (j0 + jj) * kSplitTile + 8 * t;
      act[jj] = base < vocab && bins.of(key_float(gk[jj] << 16 | 0xFFFFu)) <= cb;
#pragma unroll
      for (int v = 0; v < R; ++v)
        if (vecs) raw[jj][v] = *reinterpret_cast<const uint4*>(p + (act[jj] && base + 8 <= vocab ? base : 0) + v * (16 / sizeof(T)));
    }
  }
  uint64_t in = 0;  // this thread's logits in the bin
#pragma unroll
  for (int jj = 0; jj < kSliceTiles; ++jj) {
    if (j0 + jj >= j1) break;  // (uniform)
    uint64_t m = 0;
    if (act[jj]) {
      const int base = (j0 + jj) * kSplitTile + 8 * t;
      T e[8];
      __builtin_memcpy(e, raw[jj], sizeof(e));
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const bool ok = base + k < vocab;
        if (ok && !(vecs && base + 8 <= vocab)) e[k] = p[base + k];
        const float x = ok ? to_f32(e[k]) : -INFINITY;
        const uint64_t f = fmass(x, bins.mx);
        const int ib = f ? bins.of(x) : kPBins;
        m += ib < cb ? f : 0;
        in |= (uint64_t)(ib == cb) << (8 * jj + k);
      }
    }
    sums.add(jj, m);
  }
  for (; in; in &= in - 1) {  // (a loop over those it has, not 64 copies of the code)
    const int pos = atomicAdd(&L.n, 1);
    const int i = __builtin_ctzll(in), idx = (j0 + (i >> 3)) * kSplitTile + 8 * t + (i & 7);
    if (pos < kCandCap) st_dev_u64(pc + pos, ((uint64_t)(uint32_t)idx << 32) | fkey(to_f32(p[idx])));
  }
  sums.store(tm + j0, j1 - j0);
  if (t == 0) __hip_atomic_store(&ws.ncand[(int64_t)b * S + s], L.n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (!slice_arrive(&ws.counter[b * kCountStride], S, &L.last)) return;
  // ---- the row's last slice: all candidates
  static_assert(kMaxSplitTiles / kSliceTiles <= kSplitThreads, "a slice a thread");
  const int nc = t < S ? ld_dev(&ws.ncand[(int64_t)b * S + t]) : 0;
  uint64_t n64;
  const uint64_t upto = block_scan256((uint64_t)nc | ((uint64_t)(nc > kCandCap ? 1 : 0) << 40), L.redu, n64);
  const int n = (int)(uint32_t)n64;
  if ((n64 >> 40) || n > kPCandMax) {  // (uniform)
    if (t == 0) ws.fallback[b] = kBackBin;
    return;
  }
  if (t < S) L.off[t] = (int)(uint32_t)upto - nc;
  if (t == 0) L.off[S] = n;
  for (int j = t; j < ntiles; j += kSplitThreads) s_tile[j] = ld_dev(tm + j);
  __syncthreads();
  uint32_t diff = 0, key0 = 0;
  for (int i = t; i < n; i += kSplitThreads) {
    int lo = 0, hi = S;  // the slice whose candidates include the i-th: off[lo] <= i < off[lo + 1]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (L.off[mid] <= i) lo = mid; else hi = mid;
    }
    const uint64_t c = ld_dev(ws.cand + ((int64_t)b * S + lo) * kPBins + (i - L.off[lo]));
    L.cand[i] = c;
    if (n <= kSplitThreads) L.mass[i] = fmass(key_float((uint32_t)c), bins.mx);
  }
  if (t == 0) L.thr = 0;
  __syncthreads();
  // ---- the threshold: the largest key whose candidates at or above it, with the bins above, carry
  // `need`; each candidate against all, or over 256 of them (ties) radix selection by mass over the bits
  // in which they differ, 8 at a time
  uint32_t thr = 0;
  if (n <= kSplitThreads) {
    const Pairs pairs(n);
    const uint32_t key = (uint32_t)L.cand[min(pairs.entry(), n - 1)];
    const uint64_t f = above + pairs.mass(L.cand, L.mass, key, ~0u);
    wave_to_lds_max(&L.thr, pairs.entry() < n && f >= need ? key : 0u);
    __syncthreads();
    thr = L.thr;
  } else {
    key0 = (uint32_t)L.cand[0];
    for (int i = t; i < n; i += kSplitThreads) diff |= (uint32_t)L.cand[i] ^ key0;
    if (diff) atomicOr(&L.diff, diff);
    __syncthreads();
    diff = L.diff;
    thr = key0;
  }
  if (diff) {
    const int top = 32 - __builtin_clz(diff);
    thr = top == 32 ? 0u : key0 >> top << top;
    uint64_t acc = above;
    for (int hi = top; hi > 0;) {
      const int width = min(hi, 8), shift = hi - width;
      const uint32_t himask = hi == 32 ? 0u : ~0u << hi, nb = 1u << width;
      hi = shift;
      __syncthreads();
      L.hist[t] = 0;
      __syncthreads();
      for (int i = t; i < n; i += kSplitThreads) {
        const uint32_t key = (uint32_t)L.cand[i];
        if ((key & himask) == (thr & himask))
          atomicAdd((unsigned long long*)&L.hist[(key >> shift) & (nb - 1u)],
                    (unsigned long long)fmass(key_float(key), bins.mx));
      }
      __syncthreads();
      const uint64_t own = L.hist[kSplitThreads - 1 - t];  // (from the largest digit down)
      uint64_t sum;
      const uint64_t in = acc + block_scan256(own, L.redu, sum);
      if (in >= need && in - own < need) {
        L.bin = kSplitThreads - 1 - t;
        L.above = in - own;
      }
      __syncthreads();
      thr |= (uint32_t)L.bin << shift;
      acc = L.above;
    }
  }
  for (int i = t; i < n; i += kSplitThreads) {
    const uint64_t c = L.cand[i];
    if ((uint32_t)c >= thr)
      atomicAdd((unsigned long long*)&s_tile[(uint32_t)(c >> 32) / kSplitTile],
                (unsigned long long)fmass(key_float((uint32_t)c), bins.mx));
  }
  __syncthreads();
  pick_token(p, vocab, vec, bins.mx, thr, s_tile, ntiles, uniform[b], out + b, L.redu);
}

// ---- Top-k rows (0 < k <= kTopKMax, any top-p), one workgroup a row.  The k-th largest of the row's
// group maxima is a lower bound T0 of its k-th largest logit T* (k logits lie at or above it), and a
// close one: with 640 groups of 256 logits, about 57 logits lie above it at k = 50.  Only the groups
// whose maximum reaches T0 are read again (a tenth of the row), and their logits with key >= T0 are the
// candidates: over them, the largest T with #{key >= T} >= k is T* itself.  sample_row's rule on the
// candidates alone (T*, the top-p threshold, the inverse CDF in vocabulary order, with the same integer
// masses) gives the same token.  Where more than kTopkCands logits lie above T0 (large logits close
// together in the vocabulary), the bound is raised first.  Rows with more ties than this takes are handed
// back to sample_kernel, with the range of keys that holds T*.
constexpr int kRadixBins = 2048;  // the largest digit (11 bits) of the radix selection

constexpr int kTopkCands = 1024;  // candidates of a top-k row at most
constexpr int kPairsMax = 512;    // of which kept by the filter (all ties but 255): comparing each with all takes
                                  // 28 us a stage at 512 and 110 at 1000; a call on 1000 equal logits 160 us that way,
                                  // 32 with the one-workgroup kernel going on from the known threshold
// A top-k row whose k-th largest key lies in [lo, hi], to the one-workgroup kernel.
__device__ __forceinline__ void hand_back(const SplitWs& ws, int b, uint32_t lo, uint32_t hi) {
  ws.bin[b].above = lo;
  ws.bin[b].need = hi;
  ws.fallback[b] = kBackKeys;
}
struct TopkLds {
  union {
    int h[kRadixBins];  // (16-byte vector accesses)
    uint64_t mass[kTopkCands];
  };
  uint64_t cand[kTopkCands];  // index << 32 | key
  uint64_t sum;
  uint16_t active[kGroups];
  int wsum[kSplitThreads / kWave];
  uint32_t top, thr;  // (thr: complemented)
  int n, na, dig, above, cnt;
};

// The digit of the histogram L.h[0 .. 2048) at which the count from the top, `above` included, reaches
// k: L.dig, the count above it (L.above) and up to it (L.cnt), for every thread.
__device__ __forceinline__ void digit_select(TopkLds& L, int above, int k) {
  const int t = threadIdx.x, lane = t & (kWave - 1), wv = t / kWave;
  // thread t owns bins [8t, 8t + 8); the count in its bins and in every bin above them
  int bins[8];
  {
    const int4 a = reinterpret_cast<const int4*>(L.h)[2 * t], c = reinterpret_cast<const int4*>(L.h)[2 * t + 1];
    bins[0] = a.x; bins[1] = a.y; bins[2] = a.z; bins[3] = a.w;
    bins[4] = c.x; bins[5] = c.y; bins[6] = c.z; bins[7] = c.w;
  }
  int own = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) own += bins[e];
  int incl = own;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int v = __shfl_down(incl, o, kWave);
    incl += lane + o < kWave ? v : 0;
  }
  if (lane == 0) L.wsum[wv] = incl;
  __syncthreads();
  for (int w2 = wv + 1; w2 < kSplitThreads / kWave; ++w2) incl += L.wsum[w2];
  if (above + incl >= k && above + incl - own < k) {  // the thread whose bins hold the k-th largest
    int acc = above + incl - own;
#pragma unroll
    for (int e = 7; e >= 0; --e) {
      if (acc + bins[e] >= k) {
        L.dig = 8 * t + e;
        L.above = acc;
        L.cnt = acc + bins[e];
        break;
      }
      acc += bins[e];
    }
  }
  __syncthreads();
}
__device__ __forceinline__ void clear_hist(TopkLds& L) {
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kRadixBins / kSplitThreads / 4; ++i)
    reinterpret_cast<int4*>(L.h)[threadIdx.x * (kRadixBins / kSplitThreads / 4) + i] = make_int4(0, 0, 0, 0);
  __syncthreads();
}

// A bound that k of the row's n group maxima reach, and no more than the upper half of the k-th largest
// of them (0: fewer than k groups), and the largest of all (top), by bisection on its bits; every wave for itself, the maxima in its
// registers.
__device__ __forceinline__ uint32_t group_bound(const uint16_t* gm, int n, int k, uint32_t& top) {
  constexpr int R = kGroups / kWave / 4;
  const int lane = threadIdx.x & (kWave - 1);
  uint32_t v[kGroups / kWave];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = 4 * (r * kWave + lane);
    const uint2 u = *reinterpret_cast<const uint2*>(gm + i);
    v[4 * r] = i < n ? u.x & 0xFFFFu : 0u;
    v[4 * r + 1] = i + 1 < n ? u.x >> 16 : 0u;
    v[4 * r + 2] = i + 2 < n ? u.y & 0xFFFFu : 0u;
    v[4 * r + 3] = i + 3 < n ? u.y >> 16 : 0u;
  }
  // the bits in which some maximum differs from the largest, from the highest such bit down; a bound
  // that exactly k maxima reach is as good as the k-th largest
  uint32_t hi = 0, lo = 0xFFFFu;
#pragma unroll
  for (int r = 0; r < kGroups / kWave; ++r) {
    hi = max(hi, v[r]);
    lo = min(lo, v[r] ? v[r] : 0xFFFFu);
  }
  hi = wave_max_u32(hi);
  lo = ~wave_max_u32(~lo);
  top = hi;
  if (n < k) return 0;
  const uint32_t diff = hi ^ min(lo, hi);
  uint32_t bit = diff ? 0x80000000u >> __builtin_clz(diff) : 0u;
  uint32_t t = bit ? hi & ~(2 * bit - 1) : hi;
#pragma unroll 1
  for (; bit; bit >>= 1) {
    const uint32_t c = t | bit;
    int cnt = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (4 * r * kWave >= n) break;  // (uniform)
#pragma unroll
      for (int e = 0; e < 4; ++e) cnt += __popcll(__ballot(v[4 * r + e] >= c));
    }
    if (cnt >= k) t = c;
    if (cnt == k) break;
  }
  return t;
}

// The least logit whose key's upper half is at or above ts (ts 1: any number; a zero may be taken for
// the other one, a candidate too many).
__device__ __forceinline__ float half_key_float(uint32_t ts) { return ts <= 0x7Fu ? -INFINITY : key_float(ts << 16); }

// The token of a top-k row from its n candidates (in L.cand; at least the row's k largest): the k-th
// largest key T*, the top-p threshold over the top-k set, and the inverse CDF in vocabulary order, each by
// comparing every entry with all (Pairs; over 256 candidates, T* by radix selection).  The three stages
// share one loop: the code runs once a row, and its length is what it costs (instruction fetch).
__device__ __forceinline__ void topk_merge(int b, int n, int k, float pp, const float* uniform, int32_t* out,
                                           const SplitWs& ws, TopkLds& L) {
  const int t = threadIdx.x;
  constexpr int Q = kTopkCands / kSplitThreads;
  uint32_t most = 0;
  if (t == 0) {
    L.top = 0u;
    L.thr = 0u;
    L.sum = 0;
  }
  __syncthreads();
#pragma unroll 1
  for (int i = t; i < n; i += kSplitThreads) {
    most = max(most, (uint32_t)L.cand[i]);
    if (n <= kSplitThreads) L.mass[i] = 1;  // (counts)
  }
  wave_to_lds_max(&L.top, most);
  if (n > kSplitThreads) {
    uint32_t prefix = 0u, himask = 0u;
    int above = 0;
#pragma unroll 1
    for (int level = 0; level < 3; ++level) {  // digits of 11, 11 and 10 bits
      const int shift = level == 0 ? 21 : (level == 1 ? 10 : 0);
      const uint32_t nb = level < 2 ? 2048u : 1024u;
      clear_hist(L);
#pragma unroll 1
      for (int i = t; i < n; i += kSplitThreads) {
        const uint32_t key = (uint32_t)L.cand[i];
        if ((key & himask) == prefix) atomicAdd(&L.h[(key >> shift) & (nb - 1u)], 1);
      }
      __syncthreads();
      digit_select(L, above, k);
      prefix |= (uint32_t)L.dig << shift;
      himask |= (nb - 1u) << shift;
      above = L.above;
    }
    if (t == 0) L.thr = ~prefix;
  }
  __syncthreads();
  const float mx = key_float(L.top);
  uint32_t thr = 0;
  uint64_t need = 0, target = 0;
  int m = n;
#pragma unroll 1
  for (int stage = n > kSplitThreads ? 1 : 0; stage < 3; ++stage) {
    // 0: the entries above each; 1: at or above it; 2: kept and before it in vocabulary order
    const bool skip = stage == 1 && !(pp < 1.f);
    if (stage == 1) {
      // the top-k set, in any order: index and key, mass
      thr = ~L.thr;
      uint64_t c[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) c[q] = t + q * kSplitThreads < n ? L.cand[t + q * kSplitThreads] : 0;
      if (t == 0) L.na = 0;
      __syncthreads();
      uint64_t own = 0;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        if (t + q * kSplitThreads < n && (uint32_t)c[q] >= thr) {
          const int pos = atomicAdd(&L.na, 1);
          const uint64_t f = fmass(key_float((uint32_t)c[q]), mx);
          L.cand[pos] = c[q];
          L.mass[pos] = f;
          own += f;
        }
      }
      wave_to_lds_sum(&L.sum, own);
      if (t == 0) L.top = 0u;
      __syncthreads();
      m = L.na;
      if (m > kPairsMax) {  // (uniform)
        if (t == 0) hand_back(ws, b, thr, thr);
        return;
      }
      const uint64_t kmass = L.sum;
      const double needd = ceil((double)fmaxf(pp, 0.f) * (double)kmass);
      need = needd < 1.0 ? 1 : (uint64_t)needd;
      if (need > kmass) need = kmass;
    } else if (stage == 2) {
      // the kept mass, and where in it the uniform falls
      thr = max(thr, L.top);
      if (t == 0) L.sum = 0;
      __syncthreads();
      uint64_t own = 0;
#pragma unroll 1
      for (int e = t; e < m; e += kSplitThreads) own += (uint32_t)L.cand[e] >= thr ? L.mass[e] : 0;
      wave_to_lds_sum(&L.sum, own);
      __syncthreads();
      const uint64_t ms = L.sum;
      if (ms == 0) {  // (uniform)
        if (t == 0) out[b] = -1;
        return;
      }
      const double uu = fminf(fmaxf(uniform[b], 0.f), 1.f);
      target = (uint64_t)(uu * (double)ms);
      if (target >= ms) target = ms - 1;
    }
    const Pairs pairs(m);
    uint32_t pick = 0;
    if (!skip) {
#pragma unroll 1
      for (int e = pairs.entry(); e < (m + kSplitThreads - 1) / kSplitThreads * kSplitThreads; e += kSplitThreads) {
        const uint64_t ce = L.cand[min(e, m - 1)];
        const uint32_t key = (uint32_t)ce;
        const uint64_t f = pairs.mass(L.cand, L.mass, stage == 0 ? key + 1 : stage == 1 ? key : thr,
                                      stage == 2 ? (uint32_t)(ce >> 32) : ~0u);
        if (e < m) {
          if (stage == 0) {
            if ((int)f < k) pick = max(pick, ~key);  // (the least key with fewer than k above it)
          } else if (stage == 1) {
            if (f >= need) pick = max(pick, key);
          } else {
            const uint64_t me = key >= thr ? L.mass[e] : 0;
            if (me > 0 && f <= target && target < f + me && pairs.first()) out[b] = (int32_t)(ce >> 32);
          }
        }
      }
      if (stage < 2) wave_to_lds_max(stage == 0 ? &L.thr : &L.top, pick);
    }
    __syncthreads();
  }
}

// The row's active groups as vectors of 8 logits: item i is at base(i) in the row.
struct ActiveVectors {
  const GroupShape& g;
  const uint16_t* active;
  __device__ __forceinline__ int base(int item) const {
    const int vs = g.tg + g.gl;
    const int gi = active[item >> vs], v = item & ((1 << vs) - 1);
    const int sl = gi >> g.ps, q = (gi & (g.per_slice - 1)) << g.gl;  // (a tile group's threads from q % 256 on)
    const int tile = sl * kSliceTiles + ((q / kSplitThreads) << g.tg) + (v >> g.gl);
    return tile * kSplitTile + 8 * (q % kSplitThreads + (v & ((1 << g.gl) - 1)));
  }
};
// f(first item, x, ok) for U vectors of this thread at a time (the u-th: item first + u * kSplitThreads).
template <int U, typename T, typename F>
__device__ __forceinline__ void each_active(const T* p, int vocab, bool vec, const ActiveVectors& av, int total, F&& f) {
  constexpr int R = 8 * sizeof(T) / 16;
  const bool whole = vec && vocab >= 8;
  const int last = (vocab - 8) / 8 * 8;
#pragma unroll 1
  for (int i0 = threadIdx.x; i0 < total; i0 += U * kSplitThreads) {
    int base[U];
    uint4 raw[U][R];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int item = i0 + u * kSplitThreads;
      base[u] = item < total ? av.base(item) : vocab;
      if (whole) {
#pragma unroll
        for (int v = 0; v < R; ++v)
          raw[u][v] = *reinterpret_cast<const uint4*>(p + min(base[u], last) + v * (16 / sizeof(T)));
      }
    }
    float x[U][8];
    bool ok[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      T e[8];
      __builtin_memcpy(e, raw[u], sizeof(e));
      if (!(whole && base[u] + 8 <= vocab)) {
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (base[u] + k < vocab) e[k] = p[base[u] + k];
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        ok[u][k] = base[u] + k < vocab;
        x[u][k] = to_f32(e[k]);
      }
    }
    f(i0, x, ok);
  }
}

template <typename T>
__device__ __forceinline__ void topk_row(const T* p, int vocab, bool vec, int b, int k, float pp, const float* uniform,
                                         int32_t* out, const SplitWs& ws, TopkLds& L) {
  const int t = threadIdx.x;
  const GroupShape& g = ws.g;
  const uint16_t* gm = ws.gmax + (int64_t)b * kGroups;
  if (t == 0) L.n = L.na = 0;
  uint32_t top, ts = group_bound(gm, g.n, k, top);
  // A logit 23 or more below the largest has no mass, so it is never the token and never moves the top-p
  // threshold: the bound need not go below that (rows masked with -inf, fewer than k numbers), and fewer
  // than k candidates are then all that is kept.  (24: top is a little below the largest, and differences
  // are rounded.)
  const float least = half_key_float(top) - 24.f;
  ts = max(ts, fkey(least) >> 16);
  __syncthreads();
  for (int i = t; i < g.n; i += kSplitThreads)
    if (gm[i] >= ts) L.active[atomicAdd(&L.na, 1)] = (uint16_t)i;
  __syncthreads();
  const ActiveVectors av{g, L.active};
  const int total = L.na << (g.tg + g.gl);
#pragma unroll 1
  for (bool raised = false;; raised = true) {
    const float lim = fmaxf(half_key_float(ts), least);
    each_active<2>(p, vocab, vec, av, total, [&](int i0, const float (&x)[2][8], const bool (&ok)[2][8]) __attribute__((always_inline)) {
      uint32_t in = 0;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) in |= (uint32_t)(ok[u][e] && x[u][e] >= lim) << (8 * u + e);
      for (; in; in &= in - 1) {  // (few threads have any)
        const int pos = atomicAdd(&L.n, 1);
        const int i = __builtin_ctz(in), idx = av.base(i0 + (i >> 3) * kSplitThreads) + (i & 7);
        if (pos < kTopkCands) L.cand[pos] = ((uint64_t)(uint32_t)idx << 32) | fkey(to_f32(p[idx]));
      }
    });
    __syncthreads();
    if (raised || L.n <= kTopkCands) break;  // (uniform)
    // The start of the range of 16-bit keys (a digit of 11 bits, then one of 5) that holds the k-th
    // largest, refined until the keys at or above it fit: each level histograms, in LDS, the keys inside
    // the range chosen so far.
    const uint32_t floor_key = ts;
    uint32_t prefix = 0u, himask = 0u;
    int above = 0;
#pragma unroll 1
    for (int level = 0; level < 2; ++level) {
      const int shift = level == 0 ? 5 : 0;
      const uint32_t nb = level == 0 ? 2048u : 32u;
      clear_hist(L);
      each_active<1>(p, vocab, vec, av, total, [&](int, const float (&x)[1][8], const bool (&ok)[1][8]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t kk = ok[0][e] ? fkey(x[0][e]) >> 16 : 0u;
          if (kk >= floor_key && (kk & himask) == prefix) atomicAdd(&L.h[(kk >> shift) & (nb - 1u)], 1);
        }
      });
      if (t == 0) L.n = 0;
      __syncthreads();
      digit_select(L, above, k);
      prefix |= (uint32_t)L.dig << shift;
      himask |= (nb - 1u) << shift;
      above = L.above;
      ts = max(prefix, floor_key);
      if (L.cnt <= kTopkCands) break;  // (uniform)
    }
    if (L.cnt > kTopkCands) {  // (uniform) more than fit share the upper half of the k-th largest key
      if (t == 0) hand_back(ws, b, ts << 16, ts << 16 | 0xFFFFu);
      return;
    }
  }
  const int n = L.n;
  if (n == 0 || n > kTopkCands) {  // (uniform) no number in the row; zeros of both signs at the bound
    if (t == 0) {
      if (n == 0) out[b] = -1;
      else ws.fallback[b] = kBackRow;
    }
    return;
  }
  topk_merge(b, n, k, pp, uniform, out, ws, L);
}

template <typename T, bool WHOLE>
__global__ __launch_bounds__(kSplitThreads) __attribute__((amdgpu_waves_per_eu(5))) void split_pass_kernel(
    const T* logits, int64_t row_stride, int vocab, const int32_t* top_k, int32_t top_k_all, const float* top_p,
    float top_p_all, const float* uniform, int32_t* out, SplitWs ws) {
  union AnyLds {
    uint64_t tile[kMaxSplitTiles];
    uint64_t hist[kPBins];
    TopkLds k;
  };
  struct WholeLds {
    uint64_t tile[kMaxSplitTiles];
  };
  __shared__ __align__(16) std::conditional_t<WHOLE, WholeLds, AnyLds> L;
  __shared__ float redf[8];
  __shared__ uint64_t redu[kSliceTiles][4];
  __shared__ int s_last;
  const int s = blockIdx.x, b = blockIdx.y, S = gridDim.x;
  const int kind = WHOLE ? (int)kWholeRow : row_kind(b, vocab, top_k, top_k_all, top_p, top_p_all);
  if (kind == kOtherRow) return;
  const T* p = logits + (int64_t)b * row_stride;
  const bool vec = ((uintptr_t)p % 16) == 0;
  const int j0 = s * kSliceTiles, j1 = min(j0 + kSliceTiles, split_tiles(vocab));
  SliceLoad<T> sl;
  if constexpr (WHOLE) {
    sl.issue(p, vocab, vec, j0, j1);
    whole_slice(p, vocab, vec, sl, s, b, S, uniform, out, ws, L.tile, redf, redu, &s_last);
  } else {
    const float pp = top_p ? top_p[b] : top_p_all;
    if (kind == kTopKRow) {
      if (s == 0) topk_row(p, vocab, vec, b, top_k ? top_k[b] : top_k_all, pp, uniform, out, ws, L.k);
      return;
    }
    sl.issue(p, vocab, vec, j0, j1);
    if (kind == kWholeRow) whole_slice(p, vocab, vec, sl, s, b, S, uniform, out, ws, L.tile, redf, redu, &s_last);
    else topp_hist(p, vocab, vec, sl, s, b, S, pp, out, ws, L.hist, redf, redu[0], &s_last);
  }
}

template <typename T>
__global__ __launch_bounds__(kSplitThreads) void split_finish_kernel(const T* logits, int64_t row_stride, int vocab,
                                                                     const int32_t* top_k, int32_t top_k_all,
                                                                     const float* top_p, float top_p_all,
                                                                     const float* uniform, int32_t* out, SplitWs ws) {
  __shared__ ToppLds L;
  extern __shared__ uint64_t s_tile[];  // [ntiles]
  const int s = blockIdx.x, b = blockIdx.y;
  if (row_kind(b, vocab, top_k, top_k_all, top_p, top_p_all) == kTopPRow)
    topp_finish(logits + (int64_t)b * row_stride, vocab, s, b, gridDim.x, uniform, out, ws, L, s_tile);
}

// Which kinds of rows a call can hold (scalars settle it on the host, per-row tensors need all), and
// whether the workspace takes them over many workgroups.
struct SamplePlan {
  bool topk = true, topp = true, whole = true, other = true, whole_only = false, split = false;
  SamplePlan(int rows, int vocab, const int32_t* top_k, int32_t top_k_all, const float* top_p, float top_p_all,
             const void* ws, int64_t ws_bytes) {
    if (!top_k && !top_p) {
      const int kind = row_kind_of(top_k_all, top_p_all, vocab);
      whole = kind == kWholeRow;
      topk = kind == kTopKRow;
      topp = kind == kTopPRow;
      other = kind == kOtherRow;
    }
    whole_only = whole && !topk && !topp && !other;
    split = ws && (whole || topk || topp) && rows <= 65535 && split_tiles(vocab) <= kMaxSplitTiles &&
            ws_bytes >= split_ws_bytes(rows, vocab);
  }
};

// The launches after the scan.
template <typename T>
int launch_sample(const T* logits, int64_t row_stride, int rows, int vocab, const int32_t* top_k, int32_t top_k_all,
                  const float* top_p, float top_p_all, const float* uniform, int32_t* out, const SamplePlan& plan,
                  const SplitWs& w, hipStream_t s) {
  const dim3 grid((unsigned)split_slices(vocab), (unsigned)rows);
  if (plan.split) {
    // (top-k rows take one workgroup)
    hipLaunchKernelGGL((plan.whole_only ? split_pass_kernel<T, true> : split_pass_kernel<T, false>),
                       plan.whole || plan.topp ? grid : dim3(1, (unsigned)rows), dim3(kSplitThreads), 0, s, logits, row_stride,
                       vocab, top_k, top_k_all, top_p, top_p_all, uniform, out, w);
    if (plan.topp)
      hipLaunchKernelGGL(split_finish_kernel<T>, grid, dim3(kSplitThreads), split_tiles(vocab) * sizeof(uint64_t), s, logits, row_stride, vocab, top_k,
                         top_k_all, top_p, top_p_all, uniform, out, w);
  }
  if (!plan.split || plan.other || plan.topk || plan.topp)  // (rows may be handed back)
    hipLaunchKernelGGL(sample_kernel<T>, dim3(rows), dim3(kThreads), 0, s, logits, row_stride, vocab, top_k,
                       top_k_all, top_p, top_p_all, uniform, out, plan.split ? 1 : 0, w.fallback, w.bin);
  return (int)hipGetLastError();
}

template <typename T>
int scan_and_sample(const T* logits, int64_t row_stride, int rows, int vocab, const int32_t* top_k, int32_t top_k_all,
                    const float* top_p, float top_p_all, const float* uniform, int32_t* out, void* ws,
                    int64_t ws_bytes, hipStream_t s) {
  const SamplePlan plan(rows, vocab, top_k, top_k_all, top_p, top_p_all, ws, ws_bytes);
  SplitWs w{};
  if (plan.split) {
    w = split_ws(ws, rows, vocab);
    hipLaunchKernelGGL((plan.whole_only ? split_scan_kernel<T, false, true> : split_scan_kernel<T, false, false>), dim3((unsigned)split_slices(vocab), (unsigned)rows),
                       dim3(kSplitThreads), 0, s, logits, row_stride, vocab, top_k, top_k_all, top_p, top_p_all,
                       ScaleArgs<T>{}, w);
  }
  return launch_sample(logits, row_stride, rows, vocab, top_k, top_k_all, top_p, top_p_all, uniform, out, plan, w, s);
}

// The serving loop's scaling before sampling (ecahlang/main.py:169-170, 483-487), in one pass:
//   out[b][i] = float32(T(logits[b][i] / penalty[penalty_rows[b]][i])) / temperature[b]
// (`logits / mask_penalty` in the logits' dtype T, then `/ temperature` with a float32
// temperature, which promotes to float32).  Both divisions are IEEE divisions, as the tensor
// ops do them; a penalty or temperature of 1 leaves the value unchanged (x / 1 == x).  One
// thread per 8 logits; memory-bound.
template <typename T, bool VEC>
__global__ void scale_logits_kernel(const T* __restrict__ logits, int64_t row_stride, int vocab,
                                    const T* __restrict__ penalty, int64_t penalty_stride, int penalty_slots,
                                    const int32_t* __restrict__ penalty_rows, const float* __restrict__ temperature,
                                    float* __restrict__ out, int64_t out_stride) {
  constexpr int N = 8;  // logits per thread: 16 bytes of fp16 / bf16, two 16-byte vectors of fp32
  const int b = blockIdx.y;
  const int i0 = (blockIdx.x * blockDim.x + threadIdx.x) * N;
  if (i0 >= vocab) return;
  const T* x = logits + (int64_t)b * row_stride;
  const int prow = penalty ? penalty_rows[b] : 0;
  const T* pen = penalty ? penalty + (int64_t)prow * penalty_stride : nullptr;
  const float t = temperature ? temperature[b] : 1.f;
  float* o = out + (int64_t)b * out_stride;
  if (penalty && (prow < 0 || prow >= penalty_slots)) {  // no such penalty row: the row reads as NaN
    for (int k = 0; k < N && i0 + k < vocab; ++k) o[i0 + k] = __builtin_nanf("");
    return;
  }
  auto scale = [&](T xv, T pv) __attribute__((always_inline)) -> float {
    return scale_logit<T>(xv, pv, pen != nullptr, t);
  };
  if (VEC && i0 + N <= vocab) {
    T xs[N], ps[N];
    static_assert(N * sizeof(T) % 16 == 0, "whole 16-byte vectors");
#pragma unroll
    for (int v = 0; v < (int)(N * sizeof(T) / 16); ++v) {
      const uint4 w = *reinterpret_cast<const uint4*>(x + i0 + v * (16 / sizeof(T)));
      __builtin_memcpy(xs + v * (16 / sizeof(T)), &w, 16);
      const uint4 pw = pen ? *reinterpret_cast<const uint4*>(pen + i0 + v * (16 / sizeof(T))) : make_uint4(0, 0, 0, 0);
      __builtin_memcpy(ps + v * (16 / sizeof(T)), &pw, 16);
    }
    float ys[N];
#pragma unroll
    for (int k = 0; k < N; ++k) ys[k] = scale(xs[k], ps[k]);
#pragma unroll
    for (int v = 0; v < N / 4; ++v)
      *reinterpret_cast<float4*>(o + i0 + 4 * v) = make_float4(ys[4 * v], ys[4 * v + 1], ys[4 * v + 2], ys[4 * v + 3]);
  } else {
    for (int k = 0; k < N && i0 + k < vocab; ++k) o[i0 + k] = scale(x[i0 + k], pen ? pen[i0 + k] : from_f32<T>(1.f));
  }
}

}  // namespace

extern "C" int pkv_scale_logits(const void* logits, int64_t row_stride, int32_t rows, int32_t vocab, int32_t dtype,
                                const void* penalty, int64_t penalty_stride, int32_t penalty_slots,
                                const int32_t* penalty_rows, const float* temperature, float* out,
                                int64_t out_stride, void* stream) {
  if (rows < 0 || vocab <= 0 || row_stride < vocab || out_stride < vocab || !out) return kBadArg;
  if (penalty && (!penalty_rows || penalty_stride < vocab || penalty_slots <= 0)) return kBadArg;
  if (rows == 0) return kOk;
  if (rows > 65535) return kBadArg;
  const dim3 grid((unsigned)((vocab + 8 * 256 - 1) / (8 * 256)), (unsigned)rows);
  hipStream_t s = (hipStream_t)stream;
  const int es = dtype == kF32 ? 4 : 2;
  // 16-byte vectors when every row start is 16-byte aligned (base pointers and row strides)
  const bool vec = ((uintptr_t)logits % 16 == 0) && (row_stride * es % 16 == 0) && ((uintptr_t)out % 16 == 0) &&
                   (out_stride * 4 % 16 == 0) &&
                   (!penalty || (((uintptr_t)penalty % 16 == 0) && (penalty_stride * es % 16 == 0)));
#define PKV_SCALE(T)                                                                                          \
  do {                                                                                                        \
    if (vec)                                                                                                  \
      hipLaunchKernelGGL((scale_logits_kernel<T, true>), grid, dim3(256), 0, s, (const T*)logits, row_stride, \
                         vocab, (const T*)penalty, penalty_stride, penalty_slots, penalty_rows, temperature, out,  \
                         out_stride);                                                                         \
    else                                                                                                      \
      hipLaunchKernelGGL((scale_logits_kernel<T, false>), grid, dim3(256), 0, s, (const T*)logits, row_stride, \
                         vocab, (const T*)penalty, penalty_stride, penalty_slots, penalty_rows, temperature, out, \
                         out_stride);                                                                         \
  } while (0)
  if (dtype == kF16) PKV_SCALE(_Float16);
  else if (dtype == kBF16) PKV_SCALE(__hip_bfloat16);
  else if (dtype == kF32) PKV_SCALE(float);
  else return kBadDType;
#undef PKV_SCALE
  return (int)hipGetLastError();
}

// Whether sample_kernel takes rows of `vocab` logits of es bytes (a word of LDS per tile).
static bool row_fits(int32_t vocab, int es) { return (int64_t)vocab <= (int64_t)kMaxTiles * kThreads * (16 / es); }

static int sample_entry(const void* logits, int64_t row_stride, int32_t rows, int32_t vocab, int32_t dtype,
                        const int32_t* top_k, int32_t top_k_all, const float* top_p, float top_p_all,
                        const float* uniform, int32_t* out, void* workspace, int64_t workspace_bytes,
                        void* stream) {
  if (rows < 0 || vocab <= 0 || row_stride < vocab || !uniform || !out) return kBadArg;
  if (rows == 0) return kOk;
  const int es = dtype == kF32 ? 4 : 2;
  if (!row_fits(vocab, es)) return kBadArg;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == kF16)
    return scan_and_sample((const _Float16*)logits, row_stride, rows, vocab, top_k, top_k_all, top_p, top_p_all,
                         uniform, out, workspace, workspace_bytes, s);
  if (dtype == kBF16)
    return scan_and_sample((const __hip_bfloat16*)logits, row_stride, rows, vocab, top_k, top_k_all, top_p,
                         top_p_all, uniform, out, workspace, workspace_bytes, s);
  if (dtype == kF32)
    return scan_and_sample((const float*)logits, row_stride, rows, vocab, top_k, top_k_all, top_p, top_p_all,
                         uniform, out, workspace, workspace_bytes, s);
  return kBadDType;
}

extern "C" int pkv_top_k_top_p_sampling(const void* logits, int64_t row_stride, int32_t rows, int32_t vocab,
                                        int32_t dtype, const int32_t* top_k, int32_t top_k_all,
                                        const float* top_p, float top_p_all, const float* uniform,
                                        int32_t* out, void* stream) {
  return sample_entry(logits, row_stride, rows, vocab, dtype, top_k, top_k_all, top_p, top_p_all, uniform, out,
                      nullptr, 0, stream);
}

extern "C" int64_t pkv_sampling_workspace_bytes(int32_t rows, int32_t vocab) {
  return rows > 0 && vocab > 0 ? split_ws_bytes(rows, vocab) : 0;
}

extern "C" int pkv_top_k_top_p_sampling_ws(const void* logits, int64_t row_stride, int32_t rows, int32_t vocab,
                                           int32_t dtype, const int32_t* top_k, int32_t top_k_all,
                                           const float* top_p, float top_p_all, const float* uniform,
                                           int32_t* out, void* workspace, int64_t workspace_bytes, void* stream) {
  if (workspace && ((uintptr_t)workspace % 8)) return kBadAlign;
  return sample_entry(logits, row_stride, rows, vocab, dtype, top_k, top_k_all, top_p, top_p_all, uniform, out,
                      workspace, workspace_bytes, stream);
}

// The two calls above in one: the sampler's first pass over the logits scales them.
extern "C" int pkv_scaled_top_k_top_p_sampling(const void* logits, int64_t row_stride, int32_t rows, int32_t vocab,
                                               int32_t dtype, const void* penalty, int64_t penalty_stride,
                                               int32_t penalty_slots, const int32_t* penalty_rows,
                                               const float* temperature, float* scaled, int64_t scaled_stride,
                                               const int32_t* top_k, int32_t top_k_all, const float* top_p,
                                               float top_p_all, const float* uniform, int32_t* out, void* workspace,
                                               int64_t workspace_bytes, void* stream) {
  if (workspace && ((uintptr_t)workspace % 8)) return kBadAlign;
  if (rows < 0 || vocab <= 0 || row_stride < vocab || !uniform || !out) return kBadArg;
  if (rows == 0) return kOk;
  if (scaled_stride < vocab || !scaled) return kBadArg;
  if (penalty && (!penalty_rows || penalty_stride < vocab || penalty_slots <= 0)) return kBadArg;
  if (dtype != kF16 && dtype != kBF16 && dtype != kF32) return kBadDType;
  if (!row_fits(vocab, 4)) return kBadArg;  // (the scaled rows are fp32, whatever the logits)
  const SamplePlan plan(rows, vocab, top_k, top_k_all, top_p, top_p_all, workspace, workspace_bytes);
  // Few slices of over three tiles: the scan's workgroups would scale a slice each, a tile after the other,
  // while most of the chip is idle; scale_logits spreads the tiles (one row of 32,000 / 151,936 logits, no filter:
  // 20.8 / 21.0 us in one launch, 16.7 / 17.1 in two; 8 of 151,936, 80 slices: 22.7, 19.8; 160 slices: 23.3, 23.2;
  // 320: 30.0, 28.4; 640: 38.6, 40.1; one row of 4000, two tiles: 10.3, 11.6).
  const bool few = split_tiles(vocab) > 3 && (int64_t)rows * split_slices(vocab) <= 128;
  if (!plan.split || few || ((uintptr_t)scaled | (uintptr_t)(scaled_stride * 4)) % 16) {
    const int rc = pkv_scale_logits(logits, row_stride, rows, vocab, dtype, penalty, penalty_stride, penalty_slots,
                                    penalty_rows, temperature, scaled, scaled_stride, stream);
    return rc ? rc : sample_entry(scaled, scaled_stride, rows, vocab, kF32, top_k, top_k_all, top_p, top_p_all, uniform,
                                  out, workspace, workspace_bytes, stream);
  }
  hipStream_t s = (hipStream_t)stream;
  const SplitWs w = split_ws(workspace, rows, vocab);
  const dim3 grid((unsigned)split_slices(vocab), (unsigned)rows);
#define PKV_SCALE_SCAN(T)                                                                                          \
  hipLaunchKernelGGL((plan.whole_only ? split_scan_kernel<T, true, true> : split_scan_kernel<T, true, false>), grid, dim3(kSplitThreads), 0, s, (const T*)logits, row_stride,  \
                     vocab, top_k, top_k_all, top_p, top_p_all,                                                    \
                     (ScaleArgs<T>{(const T*)penalty, penalty_stride, penalty_slots, penalty_rows, temperature, scaled, \
                                   scaled_stride}),                                                                \
                     w)
  if (dtype == kF16) PKV_SCALE_SCAN(_Float16);
  else if (dtype == kBF16) PKV_SCALE_SCAN(__hip_bfloat16);
  else PKV_SCALE_SCAN(float);
#undef PKV_SCALE_SCAN
  return launch_sample((const float*)scaled, scaled_stride, rows, vocab, top_k, top_k_all, top_p, top_p_all, uniform, out,
                       plan, w, s);
}
