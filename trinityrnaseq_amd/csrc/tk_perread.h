// tk_perread.h -- per-read device routines shared by the single-sample
// kernels (tk_lib.hip) and the batched-component kernels (tk_batch.hip).
#pragma once
#include "tk_device.h"
#include "../../include/trinity_gpu.h"

namespace tk {

struct StatsParams {
  uint32_t min_count;
  uint32_t missing;
  int32_t nwin_policy;
  int32_t median_policy;
};

// kth smallest (0-based) of vals[0..n) by radix select over bits hb..0.
__device__ inline uint32_t wave_select(const uint32_t* vals, uint32_t n, uint32_t kth, int hb,
                                int lane) {
  uint32_t prefix = 0, pmask = 0;
  for (int bit = hb; bit >= 0; --bit) {
    uint32_t c = 0;
    for (uint32_t i = lane; i < n; i += 64) {
      const uint32_t v = vals[i];
      c += (((v & pmask) == prefix) && !((v >> bit) & 1u)) ? 1u : 0u;
    }
    c = wave_sum_u32(c);
    if (kth >= c) {
      kth -= c;
      prefix |= 1u << bit;
    }
    pmask |= 1u << bit;
  }
  return prefix;
}

// Value of one window for the coverage statistics: `has` = the window takes
// part (fastaToKmerCoverageStats.cpp skips or counts invalid windows by
// policy), v = its count, or `missing` below min_count.
__device__ __forceinline__ void window_value(const StatsParams& sp, bool in_read, bool valid, uint64_t c,
                                             bool& has, uint32_t& v) {
  has = false;
  v = 0;
  if (!in_read) return;
  if (valid) {
    v = (c != 0 && c >= sp.min_count) ? (c > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)c) : sp.missing;
    has = true;
  } else if (sp.nwin_policy == TK_NWIN_AS_MISSING) {
    v = sp.missing;
    has = true;
  }
}

// kth smallest (0-based, fewer than the values that take part) of NV values
// per lane, 0xFFFFFFFF in place of those that take no part, all below
// 2^(hb+1) otherwise: the largest value that at most kth values are below,
// bit by bit.  A step is one compare per value and scalar counting.
template <int NV>
__device__ __forceinline__ uint32_t wave_select_regs(const uint32_t (&v)[NV], uint32_t kth, int hb) {
  uint32_t prefix = 0;
  for (int bit = hb; bit >= 0; --bit) {
    const uint32_t trial = prefix | (1u << bit);
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < NV; i++) c += (uint32_t)__popcll(__ballot(v[i] < trial));
    if (c <= kth) prefix = trial;
  }
  return prefix;
}

__device__ __forceinline__ void sq_add(uint64_t v, uint64_t& lo, uint64_t& hi) {
  const uint64_t sq = v * v;
  lo += sq;
  hi += (lo < sq);
}

__device__ __forceinline__ void wave_sum_u128(uint64_t& lo, uint64_t& hi) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t ol = __shfl_xor(lo, o);
    const uint64_t oh = __shfl_xor(hi, o);
    const uint64_t nl = lo + ol;
    hi = hi + oh + (nl < lo);
    lo = nl;
  }
}

// Counts of windows base + lane and base + 64 + lane of a read (words w), as
// values x of the statistics, h where a window takes part.  Runs of at most
// 64 windows look up one key per lane.
__device__ __forceinline__ void run_values(const LaneWords& w, uint32_t base, uint32_t nwin, int k, int canonical,
                                           const TableView& t, const StatsParams& sp, uint64_t* tmp, int lane,
                                           uint32_t& xa, uint32_t& xb, bool& ha, bool& hb) {
  const uint32_t o = (uint32_t)lane & 31u, pa = base + lane, pb = pa + 64;
  uint64_t fa, fb;
  bool va, vb;
  pair_window(w.a.x, w.a.y, w.m.x, w.m.y, o, k, fa, va);
  va = va && pa < nwin;
  if (nwin <= base + 64) {
    const uint64_t keys[1] = {canon_key(fa, k, canonical)};
    const bool want[1] = {va};
    uint64_t c[1];
    coop4_get<1>(t, keys, want, tmp, lane, c);
    window_value(sp, pa < nwin, va, c[0], ha, xa);
    hb = false;
    xb = 0;
    return;
  }
  pair_window(w.b.x, w.b.y, w.m.z, w.m.w, o, k, fb, vb);
  vb = vb && pb < nwin;
  const uint64_t keys[2] = {canon_key(fa, k, canonical), canon_key(fb, k, canonical)};
  const bool want[2] = {va, vb};
  uint64_t c[2];
  coop4_get<2>(t, keys, want, tmp, lane, c);
  window_value(sp, pa < nwin, va, c[0], ha, xa);
  window_value(sp, pb < nwin, vb, c[1], hb, xb);
}

// Sums and median of NV values per lane (x[i] is 0 where h[i] is false).
template <int NV>
__device__ __forceinline__ void summarize_regs(const uint32_t (&x)[NV], const bool (&h)[NV], const StatsParams& sp,
                                               uint32_t& n, uint32_t& med, uint64_t& sum, uint64_t& sqlo,
                                               uint64_t& sqhi) {
  // while NV * 64 squares of the largest value fit 32 bits the sums take one
  // 32-bit reduction each
  constexpr uint32_t kSmall = NV == 2 ? 5792 : 4095;
  static_assert((uint64_t)kSmall * kSmall * 64 * NV < (1ull << 32), "32-bit sum of squares");
  uint32_t m = 0, v[NV];
  n = 0;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    n += (uint32_t)__popcll(__ballot(h[i]));
    m = x[i] > m ? x[i] : m;
    v[i] = h[i] ? x[i] : 0xFFFFFFFFu;
  }
  const uint32_t vmax = wave_max_u32(m);
  if (vmax <= kSmall) {
    uint32_t s = 0, q = 0;
#pragma unroll
    for (int i = 0; i < NV; i++) {
      s += x[i];
      q += (x[i] & 0xFFFFu) * (x[i] & 0xFFFFu);  // full-rate multiply
    }
    sum = wave_sum_u32(s);
    sqlo = wave_sum_u32(q);
    sqhi = 0;
  } else {
    sum = sqlo = sqhi = 0;
#pragma unroll
    for (int i = 0; i < NV; i++) {
      sum += x[i];
      sq_add(x[i], sqlo, sqhi);
    }
    sum = wave_sum_u64(sum);
    wave_sum_u128(sqlo, sqhi);
  }
  med = 0;
  if (!n) return;
  const int hb = 31 - __clz(vmax | 1u);
  if (sp.median_policy == TK_MEDIAN_LOWER) {
    med = wave_select_regs<NV>(v, (n - 1) / 2, hb);
  } else if (sp.median_policy == TK_MEDIAN_MEAN_FLOOR && !(n & 1)) {
    const uint64_t a = wave_select_regs<NV>(v, n / 2 - 1, hb);
    const uint64_t b = wave_select_regs<NV>(v, n / 2, hb);
    med = (uint32_t)((a + b) / 2);
  } else {
    med = wave_select_regs<NV>(v, n / 2, hb);
  }
}

// The statistics of a read of at most 128 * CH windows whose words start at
// wb, values in registers (two per lane and run of 128); w = its first run's
// words.
template <int CH>
__device__ __forceinline__ void stats_regs(const ReadsView& rv, uint64_t wb, LaneWords w, uint32_t nwin, int k,
                                           int canonical, const TableView& t, const StatsParams& sp, uint64_t* tmp,
                                           int lane, uint32_t& n, uint32_t& med, uint64_t& sum, uint64_t& sqlo,
                                           uint64_t& sqhi) {
  uint32_t x[2 * CH];
  bool h[2 * CH];
#pragma unroll
  for (int c = 0; c < CH; c++) {
    const uint32_t base = 128 * c;
    LaneWords next = w;
    if (c + 1 < CH && base + 128 < nwin) next = lane_words(rv, wb + 4 * (c + 1), lane);
    x[2 * c] = x[2 * c + 1] = 0;
    h[2 * c] = h[2 * c + 1] = false;
    if (c == 0 || base < nwin)
      run_values(w, base, nwin, k, canonical, t, sp, tmp, lane, x[2 * c], x[2 * c + 1], h[2 * c], h[2 * c + 1]);
    w = next;
  }
  summarize_regs<2 * CH>(x, h, sp, n, med, sum, sqlo, sqhi);
}

__device__ __forceinline__ void write_stat(int lane, uint32_t med, uint32_t n, uint64_t sum, uint64_t sqlo,
                                           uint64_t sqhi, tk_read_stat* out) {
  if (lane == 0) {
    tk_read_stat st;
    st.median = med;
    st.nwin = n;
    st.sum = sum;
    st.sumsq_lo = sqlo;
    st.sumsq_hi = sqhi;
    *out = st;
  }
}

// fastaToKmerCoverageStats for read r, one wavefront: exact integer sums and
// the median by radix select.  Reads of up to 128 windows keep their values
// in registers (two per lane); longer reads stage them in `vals` (LDS, >=
// nwin entries) 128 windows at a time.  tmp: kLookupScratch u64 of LDS for the
// cooperative lookup.  Lane 0 writes *out.
// kShortOnly: the caller guarantees nwin <= 128 (the long-read path is not
// compiled, which frees registers).
template <bool kShortOnly = false>
__device__ inline void stats_read(const ReadsView& rv, uint64_t r, int k, int canonical,
                                  const TableView& t, const StatsParams& sp, uint32_t* vals,
                                  uint64_t* tmp, int lane, tk_read_stat* out) {
  const uint32_t L = rv.len[r];
  const uint32_t nwin = L >= (uint32_t)k ? L - k + 1 : 0;
  const uint64_t wb = rv.word_off[r];
  uint32_t n = 0, vmax = 0, med = 0;
  uint64_t sum = 0, sqlo = 0, sqhi = 0;
  if (kShortOnly || nwin <= 128) {
    stats_regs<1>(rv, wb, lane_words(rv, wb, lane), nwin, k, canonical, t, sp, tmp, lane, n, med, sum, sqlo, sqhi);
  } else {
    // windows are taken 128 at a time (two per lane), values appended to
    // vals in window order
    for (uint32_t base = 0; base < nwin; base += 128) {
      uint32_t x[2];
      bool h[2];
      run_values(lane_words(rv, wb + base / 32, lane), base, nwin, k, canonical, t, sp, tmp, lane, x[0], x[1], h[0],
                 h[1]);
#pragma unroll
      for (int half = 0; half < 2; half++) {
        const uint64_t m = __ballot(h[half]);
        if (h[half]) {
          const uint32_t v = x[half];
          vals[n + __popcll(m & ((1ull << lane) - 1))] = v;
          sum += v;
          sq_add(v, sqlo, sqhi);
          vmax = v > vmax ? v : vmax;
        }
        n += (uint32_t)__popcll(m);
      }
    }
    wave_sync();
    sum = wave_sum_u64(sum);
    wave_sum_u128(sqlo, sqhi);
    if (n) {
      vmax = wave_max_u32(vmax);
      const int hb = 31 - __clz(vmax | 1u);
      if (sp.median_policy == TK_MEDIAN_LOWER) {
        med = wave_select(vals, n, (n - 1) / 2, hb, lane);
      } else if (sp.median_policy == TK_MEDIAN_MEAN_FLOOR && !(n & 1)) {
        const uint64_t a = wave_select(vals, n, n / 2 - 1, hb, lane);
        const uint64_t b = wave_select(vals, n, n / 2, hb, lane);
        med = (uint32_t)((a + b) / 2);
      } else {
        med = wave_select(vals, n, n / 2, hb, lane);
      }
    }
  }
  write_stat(lane, med, n, sum, sqlo, sqhi, out);
  wave_sync();
}

// Block-shared LDS cache of table counts (tagged key -> count), for reads
// taken in the locality order: a read's windows are mostly its
// predecessors', so the block looks a key up in HBM once and its later reads
// find it here.  A slot's key is claimed by CAS and its value written after;
// a reader that finds the key before the value (kNotReady) treats it as a
// miss, so a lookup never returns a wrong count.  Slots are never reused.
constexpr uint32_t kNotReady = 0xFFFFFFFFu;
constexpr int kCacheProbe = 16;

struct CountCache {
  uint64_t* keys;   // 0 = empty
  uint32_t* vals;   // kNotReady until written
  uint32_t mask;    // slots - 1
};

__device__ __forceinline__ uint32_t cache_home(uint64_t tagged, uint32_t mask) {
  return (uint32_t)((tagged * 0x9E3779B97F4A7C15ULL) >> 40) & mask;
}

__device__ __forceinline__ bool cache_get(const CountCache& c, uint64_t tagged, uint32_t& v) {
  uint32_t h = cache_home(tagged, c.mask);
  for (int p = 0; p < kCacheProbe; p++) {
    const uint64_t k = c.keys[h];
    if (k == tagged) {
      v = c.vals[h];
      return v != kNotReady;
    }
    if (k == 0) return false;
    h = (h + 1) & c.mask;
  }
  return false;
}

__device__ __forceinline__ void cache_put(const CountCache& c, uint64_t tagged, uint32_t v) {
  uint32_t h = cache_home(tagged, c.mask);
  for (int p = 0; p < kCacheProbe; p++) {
    uint64_t k = c.keys[h];
    if (k == 0) {
      k = atomicCAS((unsigned long long*)&c.keys[h], 0ULL, (unsigned long long)tagged);
      if (k == 0) {
        c.vals[h] = v;
        return;
      }
    }
    if (k == tagged) return;
    h = (h + 1) & c.mask;
  }
}

// stats_read for a read of at most 128 windows, with the block's count
// cache in front of the table: only keys the cache does not hold are looked
// up (the others' lanes load bucket 0 with them), and those are added to it.
__device__ inline void stats_read_cached(const ReadsView& rv, uint64_t r, int k, int canonical,
                                         const TableView& t, const StatsParams& sp, const CountCache& cc,
                                         uint64_t* tmp, int lane, tk_read_stat* out) {
  const uint32_t L = rv.len[r];
  const uint32_t nwin = L >= (uint32_t)k ? L - k + 1 : 0;
  const uint64_t wb = rv.word_off[r];
  const uint32_t pa = lane, pb = 64 + lane;
  uint64_t fa = 0, fb = 0;
  bool va = false, vb = false;
  if (pa < nwin) window_at(rv, wb, pa, k, fa, va);
  if (pb < nwin) window_at(rv, wb, pb, k, fb, vb);
  const uint64_t keys[2] = {va ? canon_key(fa, k, canonical) : 0, vb ? canon_key(fb, k, canonical) : 0};
  uint32_t cva = 0, cvb = 0;
  const bool hita = va && cache_get(cc, keys[0] | t.occ, cva);
  const bool hitb = vb && cache_get(cc, keys[1] | t.occ, cvb);
  const bool want[2] = {va && !hita, vb && !hitb};
  uint64_t c[2];
  coop4_get<2>(t, keys, want, tmp, lane, c);
  if (want[0] && c[0] < kNotReady) cache_put(cc, keys[0] | t.occ, (uint32_t)c[0]);
  if (want[1] && c[1] < kNotReady) cache_put(cc, keys[1] | t.occ, (uint32_t)c[1]);
  if (hita) c[0] = cva;
  if (hitb) c[1] = cvb;
  bool h[2];
  uint32_t x[2];
  window_value(sp, pa < nwin, va, c[0], h[0], x[0]);
  window_value(sp, pb < nwin, vb, c[1], h[1], x[1]);
  uint32_t n, med;
  uint64_t sum, sqlo, sqhi;
  summarize_regs<2>(x, h, sp, n, med, sum, sqlo, sqhi);
  write_stat(lane, med, n, sum, sqlo, sqhi, out);
  wave_sync();
}

// Component table: 64-byte buckets of four 16-byte slots (tagged key, ~comp);
// buckets [boff, boff + bmask] belong to one table.  A key's probe sequence
// wraps within its region of 1024 buckets (half full over its 4096 or 8192
// slots), so a region can be built apart from the others (k_batch_ctable_lds).
constexpr uint32_t kCtRegionBits = 10;
constexpr uint64_t kCtRegion = 1ull << kCtRegionBits;

__device__ __forceinline__ uint64_t ct_rmask(uint64_t bmask) { return bmask < kCtRegion ? bmask : kCtRegion - 1; }
__device__ __forceinline__ uint64_t ct_next(uint64_t b, uint64_t rmask) { return (b & ~rmask) | ((b + 1) & rmask); }

__device__ inline void ctable_add(uint64_t* slots, uint64_t boff, uint64_t bmask, uint64_t occ,
                                  uint64_t key, uint32_t comp, uint32_t& mynew, uint32_t* err) {
  const uint64_t tagged = key | occ;
  const uint64_t rmask = ct_rmask(bmask);
  uint64_t b = mix64(key) & bmask;
  for (uint64_t p = 0; p <= rmask; p++) {
    uint64_t* line = slots + ((boff + b) << 3);
    for (int j = 0; j < 4; j++) {
      uint64_t s = line[2 * j];
      if (s == 0) {
        s = atomicCAS((unsigned long long*)&line[2 * j], 0ULL, (unsigned long long)tagged);
        if (s == 0) { mynew++; s = tagged; }
      }
      if (s == tagged) {
        // a value seen is never above the slot's: it only grows
        if ((uint32_t)line[2 * j + 1] < ~comp) atomicMax((unsigned int*)&line[2 * j + 1], ~comp);
        return;
      }
    }
    b = ct_next(b, rmask);
  }
  atomicOr(err, 1u);
}

// Packed component table (k <= 25): 64-byte buckets of eight 8-byte slots
// [vmax - comp : 63-2k | occupied : 1 | key : 2k], vmax = 2^(63-2k) - 1, so
// a new key costs one CAS and the largest word of one key holds its
// smallest comp; comp <= vmax.
__device__ inline void pctable_put(uint64_t* slots, uint64_t boff, uint64_t bmask, int k, uint64_t word,
                                   uint32_t* err) {
  const uint64_t occ = 1ull << (2 * k), km = (occ << 1) - 1, tagged = word & km;
  const uint64_t rmask = ct_rmask(bmask);
  uint64_t b = mix64(word & (occ - 1)) & bmask;
  for (uint64_t p = 0; p <= rmask; p++) {
    uint64_t* line = slots + ((boff + b) << 3);
    for (int j = 0; j < 8; j++) {
      uint64_t s = line[j];
      if (s == 0) {
        s = atomicCAS((unsigned long long*)&line[j], 0ULL, (unsigned long long)word);
        if (s == 0) return;
      }
      if ((s & km) == tagged) {
        if (s < word) atomicMax((unsigned long long*)&line[j], (unsigned long long)word);
        return;
      }
    }
    b = ct_next(b, rmask);
  }
  atomicOr(err, 1u);
}

__device__ inline void pctable_add(uint64_t* slots, uint64_t boff, uint64_t bmask, int k, uint64_t key,
                                   uint32_t comp, uint32_t* err) {
  const uint64_t vmax = (1ull << (63 - 2 * k)) - 1;
  pctable_put(slots, boff, bmask, k, ((vmax - comp) << (2 * k + 1)) | (1ull << (2 * k)) | key, err);
}

__device__ __forceinline__ uint32_t pctable_comp(uint64_t s, int k) {
  return (uint32_t)(((1ull << (63 - 2 * k)) - 1) - (s >> (2 * k + 1)));
}

// Component tables for coop_lookup: the value is the component (kNone, above
// every 32-bit id, when absent).
struct CtLayout {  // four two-word slots, one per lane
  static constexpr uint64_t kNone = 1ull << 32;
  __device__ __forceinline__ bool match(const ulonglong2& s, uint64_t tag, uint64_t& v) const {
    v = (uint32_t)~s.y;
    return s.x == tag;
  }
  static __device__ __forceinline__ bool full(const ulonglong2& s) { return s.x != 0; }
};
struct PtLayout {  // eight one-word slots, two per lane
  static constexpr uint64_t kNone = 1ull << 32;
  uint64_t km;
  int k;
  __device__ __forceinline__ bool match(const ulonglong2& s, uint64_t tag, uint64_t& v) const {
    const bool m0 = (s.x & km) == tag, m1 = (s.y & km) == tag;
    v = pctable_comp(m0 ? s.x : s.y, k);
    return m0 | m1;
  }
  static __device__ __forceinline__ bool full(const ulonglong2& s) { return s.y != 0; }
};

// Component of a key whose home bucket is full and does not hold it: the
// buckets after it, as table_field_after.
template <class L>
__device__ __forceinline__ uint64_t comp_after(const uint64_t* slots, uint64_t boff, uint64_t bmask, const L& lay,
                                               uint64_t key, uint64_t tag) {
  const uint64_t rmask = ct_rmask(bmask);
  uint64_t b = mix64(key) & bmask;
  for (uint64_t p = 1; p <= rmask; p++) {
    b = ct_next(b, rmask);
    const ulonglong2* l2 = reinterpret_cast<const ulonglong2*>(slots + ((boff + b) << 3));
    const ulonglong2 v[4] = {l2[0], l2[1], l2[2], l2[3]};
    uint64_t res = L::kNone, x;
#pragma unroll
    for (int j = 0; j < 4; j++) res = lay.match(v[j], tag, x) ? x : res;
    if (res != L::kNone || !L::full(v[3])) return res;
  }
  return L::kNone;
}

// Components of the keys, NK per lane (0xFFFFFFFF = absent or want[i] false).
template <bool kPacked, int NK>
__device__ __forceinline__ void coop_comps(const uint64_t* slots, uint64_t boff, uint64_t bmask, int k,
                                           const uint64_t (&key)[NK], const bool (&want)[NK], uint64_t* scratch,
                                           int lane, uint32_t (&comp)[NK]) {
  const uint64_t occ = 1ull << (2 * k);
  uint64_t off[NK], tag[NK], out[NK];
#pragma unroll
  for (int i = 0; i < NK; i++) {
    off[i] = want[i] ? (boff + (mix64(key[i]) & bmask)) << 6 : 0;
    tag[i] = want[i] ? key[i] | occ : 0;
  }
  const auto lay = [&] {
    if constexpr (kPacked) return PtLayout{(occ << 1) - 1, k};
    else return CtLayout{};
  }();
  coop_lookup<NK>(slots, lay, off, tag, scratch, lane, out);
#pragma unroll
  for (int i = 0; i < NK; i++) {
    if (want[i] && out[i] == kLookupFull) out[i] = comp_after(slots, boff, bmask, lay, key[i], tag[i]);
    comp[i] = want[i] && out[i] < (1ull << 32) ? (uint32_t)out[i] : 0xFFFFFFFFu;
  }
}

// The component with most of NV votes per lane (0xFFFFFFFF = no vote) and its
// votes: the distinct components in ascending order, the first strictly
// largest count wins (ties -> smallest id); no vote left can win once they are
// no more than the best has.
template <int NV>
__device__ __forceinline__ void vote_regs(uint32_t (&c)[NV], uint32_t& best, uint32_t& bestn) {
  best = 0xFFFFFFFFu;
  bestn = 0;
  uint32_t left = 0;
#pragma unroll
  for (int i = 0; i < NV; i++) left += (uint32_t)__popcll(__ballot(c[i] != 0xFFFFFFFFu));
  while (left > bestn) {
    uint32_t m = c[0];
#pragma unroll
    for (int i = 1; i < NV; i++) m = c[i] < m ? c[i] : m;
    const uint32_t cand = wave_min_u32(m);
    uint32_t cnt = 0;
#pragma unroll
    for (int i = 0; i < NV; i++) {
      const bool is = c[i] == cand;
      cnt += (uint32_t)__popcll(__ballot(is));
      c[i] = is ? 0xFFFFFFFFu : c[i];
    }
    left -= cnt;
    if (cnt > bestn) {
      bestn = cnt;
      best = cand;
    }
  }
}

// Components of windows base + lane and base + 64 + lane of a read (words w),
// one key per lane at a time: the registers of two would cost two of the seven
// waves per SIMD that hide the misses (6 M reads: 10.2 ms with two).
template <bool kPacked>
__device__ __forceinline__ void run_comps(const LaneWords& w, uint32_t base, uint32_t nwin, int k, int canonical,
                                          const uint64_t* slots, uint64_t boff, uint64_t bmask, uint64_t* scratch,
                                          int lane, uint32_t (&c)[2]) {
  const uint32_t o = (uint32_t)lane & 31u;
  words2 x = w.a;
  uint32_t mx = w.m.x, my = w.m.y;
  c[0] = c[1] = 0xFFFFFFFFu;
#pragma unroll 1
  for (uint32_t p = base; p < nwin && p < base + 128; p += 64) {
    uint64_t f;
    bool v;
    pair_window(x.x, x.y, mx, my, o, k, f, v);
    const uint64_t keys[1] = {canon_key(f, k, canonical)};
    const bool want[1] = {v && p + lane < nwin};
    uint32_t one[1];
    coop_comps<kPacked, 1>(slots, boff, bmask, k, keys, want, scratch, lane, one);
    c[1] = c[0];  // which is which does not matter to the vote
    c[0] = one[0];
    x = w.b;
    mx = w.m.z;
    my = w.m.w;
  }
}

__device__ __forceinline__ void write_vote(int lane, uint32_t best, uint32_t bestn, uint32_t nwin, tk_r2t_vote* out) {
  if (lane == 0) {
    tk_r2t_vote v;
    v.comp = best;
    v.hits = bestn;
    v.nwin = nwin;
    *out = v;
  }
}

// ReadsToTranscripts vote of read r, one wavefront.  Reads of at most 128
// windows vote from registers; longer ones stage the component ids of their
// hitting windows in `hits` (LDS) and walk the distinct ids in ascending
// order.  kPacked: the component table is the packed layout (pctable_add).
// scratch: kLookupScratch u64 of LDS.
template <bool kPacked = false>
__device__ inline void vote_read(const ReadsView& rv, uint64_t r, int k, int canonical,
                                 const uint64_t* slots, uint64_t boff, uint64_t bmask,
                                 uint32_t* hits, uint64_t* scratch, int lane, tk_r2t_vote* out) {
  const uint32_t L = rv.len[r];
  const uint32_t nwin = L >= (uint32_t)k ? L - k + 1 : 0;
  const uint64_t wb = rv.word_off[r];
  uint32_t best = 0xFFFFFFFFu, bestn = 0;
  uint32_t c[2];
  if (nwin <= 128) {
    run_comps<kPacked>(lane_words(rv, wb, lane), 0, nwin, k, canonical, slots, boff, bmask, scratch, lane, c);
    vote_regs<2>(c, best, bestn);
  } else {
    uint32_t n = 0;
    for (uint32_t base = 0; base < nwin; base += 128) {
      run_comps<kPacked>(lane_words(rv, wb + base / 32, lane), base, nwin, k, canonical, slots, boff, bmask, scratch,
                         lane, c);
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const bool has = c[i] != 0xFFFFFFFFu;
        const uint64_t m = __ballot(has);
        if (has) hits[n + __popcll(m & ((1ull << lane) - 1))] = c[i];
        n += (uint32_t)__popcll(m);
      }
    }
    wave_sync();
    uint32_t prev = 0, left = n;
    bool first = true;
    while (left > bestn) {
      uint32_t cand = 0xFFFFFFFFu;
      for (uint32_t i = lane; i < n; i += 64) {
        const uint32_t v = hits[i];
        if ((first || v > prev) && v < cand) cand = v;
      }
      cand = wave_min_u32(cand);
      uint32_t cnt = 0;
      for (uint32_t i = lane; i < n; i += 64) cnt += hits[i] == cand;
      cnt = wave_sum_u32(cnt);
      left -= cnt;
      if (cnt > bestn) {
        bestn = cnt;
        best = cand;
      }
      prev = cand;
      first = false;
    }
  }
  write_vote(lane, best, bestn, nwin, out);
  wave_sync();
}

}  // namespace tk
