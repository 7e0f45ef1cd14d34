// tk_count_agg.h -- the block-merging count pass (k_count_agg), shared by
// the single-table count (tk_lib.hip) and the batched components
// (tk_batch.hip), whose blocks each merge one component's reads.
#pragma once
#include <algorithm>

#include "tk_device.h"

namespace tk {

constexpr int kReadsPerBlock = 64;

// Block-aggregated count for reads taken in the locality order, where the
// 64 reads of a group largely overlap one locus.  Every device-scope atomic
// on the table is a round trip to the memory side (the eight XCDs' L2s are
// not coherent with each other), so the count pass is bound by the number
// of atomics, not by bytes: the block first merges its windows in an LDS hash
// table of words `tagged key | occurrences << (2k+1)` (the global slot
// format), and only when the table could pass 3/4 load (or a count kMaxRun)
// does each distinct key reach the global table, once, with its number of
// occurrences, through the cooperative four-lane add.  Needs cmax >= kMaxRun
// (k <= 25), so neither the LDS word nor one global add carries more than once.
//
// The merge is bound by vector instruction issue (70% of the cycles, 125
// instructions per 64 windows; 69% and 222 with the bucketed table and two
// windows per lane and barrier it had before, where a wave ran every probe step
// until its unluckiest lane was done).  So the lanes run free of each other: a step probes one
// slot per lane (a CAS of the window's word; slots are single)
// and a lane whose window is in rolls to its next one in the same step, about
// 1.5 steps per window whatever the others need.  Four threads per read, each
// rolling over a quarter of its windows.  A round is as many steps as the
// table has room for; one barrier and one LDS add per wave and round tell every
// thread the new keys, the windows merged and whether any lane has work left.
// 5.04 G windows of 150-base reads (EMIT): 35.9 -> 23.3 ms, 216 G windows/s;
// 2 M pairs 4.22 -> 2.60 ms; with table atomics, which bound that form, 14.5 ->
// 13.6 ms.  Tables of 4,864 slots, four blocks per CU instead of five: 25.2 ms.
//
// EMIT: instead of adding them to the table, a flush appends the block's
// merged words to `out` for the region-resident passes below.  The grid is
// then persistent (each block takes groups of 64 reads grid-stride, keeps its
// table over the groups, and loads the next group's reads while it merges) and
// a wavefront reserves the stream `chunk` words at a time (chunk >= SLOTS / 4,
// the most one of its flushes emits), so the shared cursor sees one atomic per
// chunk, not one per flush.  A flush that does not fit below `cap` is added to
// the table; every reserved word below `cap` that holds no merged word is
// zero, so out[0, min(*cursor, cap)) is always defined (0 = no word).
//
// Groups says which reads a block merges and into which table: count() groups,
// get(g, r0, nr, t) gives group g's first position r0 in the read order, its
// nr <= kReadsPerBlock reads and the table its flushes add to (every table of
// one pass has the same key and count layout).
//
// KHI (k >= 17): a base enters and leaves the k-mers in their high words, so
// the low ones need no masks.

// Home slot of a key in the LDS table, below SLOTS (the factors are kept below
// 2^24, where a multiply runs at full rate; in unsigned arithmetic throughout).
template <int SLOTS>
__device__ __forceinline__ uint32_t agg_home(uint32_t lo, uint32_t hi) {
  const uint32_t x = (lo ^ (lo >> 15) ^ (hi << 7)) & 0xFFFFFFu;
  const uint32_t h = (x * 0x9E3779u) >> 16;  // 16 bits
  return (h * (uint32_t)SLOTS) >> 16;
}

// Probe stride of a key: 1, 7, 11 or 13, none of which shares a factor with
// SLOTS (2^a 3^b 5^c), so every probe sequence visits every slot.  Against
// linear probing the four sequences cut a fifth of the steps near 3/4 load.
__device__ __forceinline__ uint32_t agg_stride(uint32_t lo) { return (0x0D0B0701u >> (lo & 24u)) & 0xFFu; }

template <int SLOTS, bool EMIT, bool KHI, class Groups>
__device__ __forceinline__ void count_agg(ReadsView rv, const Groups& groups, int k, int canonical, TableView t,
                                          uint32_t* __restrict__ flags, uint64_t* __restrict__ out, uint64_t cap,
                                          uint64_t chunk, unsigned long long* __restrict__ cursor,
                                          int table_ok = 1) {
  extern __shared__ uint64_t s_tab[];  // SLOTS words, 0 = empty
  __shared__ uint32_t s_round[3];      // this round's sums, the next one's, and the one being cleared
  __shared__ uint32_t s_new;
  constexpr uint32_t kMaxDistinct = SLOTS / 4 * 3;  // LDS load <= 3/4
  constexpr uint32_t kMaxRun = 8064;                // occurrences per merge <= cmax (k <= 25)
  constexpr uint32_t kQuarter = SLOTS / 4;
  constexpr uint32_t kMaxSteps = 8;  // per round: the sums below fit 12 bits each
  // Steps a round must have room for; with less the table is flushed.  Fewer
  // barriers against fewer windows per word: the stream's words are cheap (5.04 G
  // windows: 27.9 ms at 1, 24.9 at 2, 23.3 at 3, the passes behind it +0.8 ms in
  // all), the table's atomics are not.
  constexpr uint32_t kMinSteps = EMIT ? 3 : 1;
  static_assert(SLOTS == 3840 || SLOTS == 4096, "slots coprime to the strides");
  static_assert(kQuarter % 64 == 0 && kMaxDistinct >= 256 && 256 * kMaxSteps < 4096, "round sums");
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint64_t ngroups = groups.count();
  const uint64_t g0 = EMIT ? blockIdx.x : xcd_block(blockIdx.x, gridDim.x);
  const uint64_t gstride = EMIT ? gridDim.x : ngroups;
  for (int i = tid; i < SLOTS; i += blockDim.x) s_tab[i] = 0;
  if (tid < 3) s_round[tid] = 0;
  if (tid == 0) s_new = 0;
  __syncthreads();
  const uint64_t one = 1ull << t.cshift;
  const uint64_t kmask = (1ull << (2 * k)) - 1;
  const uint32_t mhi = (uint32_t)(kmask >> 32), rsh = (uint32_t)(2 * k - 2);
  const uint32_t khi = (uint32_t)(t.kmo >> 32);
  uint64_t* quarter = s_tab + (uint32_t)wv * kQuarter;
  uint32_t mynew = 0;
  uint64_t cur = 0, cend = 0;  // the wave's reserved chunk of the stream
  uint32_t distinct = 0, since = 0, par = 0;  // block-uniform
  const int rj = tid >> 2;
  const uint32_t rp = (uint32_t)tid & 3u;

  // Every wavefront takes its quarter of the table out and clears it; the
  // caller has passed a barrier since the last insert.
  auto flush = [&]() {
    if (EMIT) {
      constexpr int kPer = kQuarter / 64;
      uint64_t v[kPer];
      uint32_t nd = 0;
#pragma unroll
      for (int i = 0; i < kPer; i++) v[i] = quarter[64 * i + lane];
#pragma unroll
      for (int i = 0; i < kPer; i++) nd += (uint32_t)__popcll(__ballot(v[i] != 0));
      if (cur + nd > cend) {
        const uint64_t z1 = cend < cap ? cend : cap;
        for (uint64_t i = cur + lane; i < z1; i += 64) out[i] = 0;
        unsigned long long c = 0;
        if (lane == 0) c = atomicAdd(cursor, (unsigned long long)chunk);
        cur = __shfl(c, 0);
        cend = cur + chunk;
      }
      if (cur + nd <= (cend < cap ? cend : cap)) {
        uint64_t at = cur;
#pragma unroll
        for (int i = 0; i < kPer; i++) {
          const uint64_t m = __ballot(v[i] != 0);
          if (v[i]) out[at + (uint32_t)__popcll(m & ((1ull << lane) - 1))] = v[i];
          at += (uint32_t)__popcll(m);
        }
        cur = at;
      } else if (!table_ok) {
        // the table is not yet cleared: such a flush is dropped and flags[6]
        // set; the caller clears the table and merges again
        if (lane == 0 && nd) atomicOr(&flags[6], 1u);
      } else {
        for (uint32_t i = lane; i < kQuarter; i += 64) {
          const uint64_t w = quarter[i];
          if (!w) continue;
          const uint32_t r = table_add(t, w & (t.occ - 1), w >> t.cshift, &flags[0]);
          if (r == 2u) atomicOr(&flags[0], 1u);
          else mynew += r;
        }
      }
      for (uint32_t i = lane; i < kQuarter; i += 64) quarter[i] = 0;
    } else {
      // compact the quarter in place (a wavefront's LDS reads of a batch
      // precede its writes, and writes land at or below the batch being
      // read), then add 64 keys at a time
      uint32_t nd = 0;
      for (uint32_t i0 = 0; i0 < kQuarter; i0 += 64) {
        const uint64_t v = quarter[i0 + lane];
        const uint64_t m = __ballot(v != 0);
        if (v) quarter[nd + (uint32_t)__popcll(m & ((1ull << lane) - 1))] = v;
        nd += (uint32_t)__popcll(m);
      }
      wave_sync();
      for (uint32_t e0 = 0; e0 < nd; e0 += 64) {
        const bool want = e0 + lane < nd;
        const uint64_t v = want ? quarter[e0 + lane] : 0;
        bool lost = false;
        mynew += coop4_add(t, v & (t.occ - 1), want, lane, &flags[0], lost, want ? v >> t.cshift : 1);
        if (lost) atomicOr(&flags[0], 1u);
      }
      wave_sync();
      for (uint32_t i = lane; i < kQuarter; i += 64) quarter[i] = 0;
    }
    distinct = since = 0;
    __syncthreads();
  };

  // this thread's read of a group: its length and first word
  uint32_t L = 0;
  uint64_t wb = 0;
  auto fetch = [&](uint64_t grp, TableView& tt, uint64_t& r) {
    uint64_t r0 = 0;
    int nr = 0;
    if (grp < ngroups) groups.get(grp, r0, nr, tt);
    const bool have = rj < nr;
    if (have) r = read_at(rv, r0 + rj);
    return have;
  };
  {
    uint64_t r = 0;
    if (fetch(g0, t, r)) {
      L = rv.len[r];
      wb = rv.word_off[r];
    }
  }
  for (uint64_t grp = g0; grp < ngroups; grp += gstride) {
    const uint32_t nw = L >= (uint32_t)k ? L - k + 1 : 0;
    const uint32_t q = (nw + 3) >> 2;
    const uint32_t rs = min(nw, rp * q);
    uint32_t rem = min(nw, rs + q) - rs;  // windows not yet begun
    // words rs/32 .. rs/32 + 2: a quarter of up to 32 windows needs no more
    uint64_t c0 = 0, c1 = 0, nxt = 0;
    uint32_t m0 = 0, m1 = 0, nm = 0, wnext = rs >> 5;
    if (rem) {
      c0 = rv.codes[wb + wnext];
      c1 = rv.codes[wb + wnext + 1];
      nxt = rv.codes[wb + wnext + 2];
      m0 = rv.nmask[wb + wnext];
      m1 = rv.nmask[wb + wnext + 1];
      nm = rv.nmask[wb + wnext + 2];
    }
    // the next group's read, loaded in two steps between the rounds
    uint64_t nr_ = 0, nwb = 0;
    uint32_t nL = 0;
    bool nhave = false;
    if (EMIT) {
      TableView same = t;
      nhave = fetch(grp + gstride, same, nr_);
    }
    int stage = 0;
    // first window, and the rolling state after it: k-mer words (f, r), the
    // current code word shifted so that the next base sits in its top bits
    uint64_t fwd = 0, rcm = 0, cw = 0;
    uint32_t cm = 0, run = 0, left = 0;
    bool pend = false;
    uint64_t word = 0;
    uint32_t idx = 0;
    auto take = [&]() {  // the window (fwd, rcm) becomes the lane's pending word
      const uint64_t tagged = ((canonical && rcm < fwd) ? rcm : fwd);
      idx = agg_home<SLOTS>((uint32_t)tagged, (uint32_t)(tagged >> 32));
      word = tagged | t.occ | one;
    };
    if (rem) {
      const uint32_t o = rs & 31u;
      const uint64_t x = (c0 << (2 * o)) | ((c1 >> 1) >> (63 - 2 * o));
      const uint32_t mw = (m0 << o) | ((m1 >> 1) >> (31 - o));
      fwd = x >> (64 - 2 * k);
      const uint32_t nmk = mw >> (32 - k);
      rcm = revcomp(fwd, k);
      run = nmk ? (uint32_t)__builtin_ctz(nmk) : (uint32_t)k;
      // the next base, rs + k, is in word rs/32 or rs/32 + 1 (k <= 25)
      const uint32_t pos = rs + k, po = pos & 31u;
      const bool second = (pos >> 5) != (rs >> 5);
      cw = (second ? c1 : c0) << (2 * po);
      cm = (second ? m1 : m0) << po;
      if (!second) {
        nxt = c1;
        nm = m1;
      }
      wnext = (pos >> 5) + 2;
      left = 32 - po;
      rem--;
      pend = run >= (uint32_t)k;
      take();
    }
    const bool last = grp + gstride >= ngroups;
    bool done = false;  // this group's windows are in
    for (;;) {
      uint32_t steps = min((kMaxDistinct - distinct) >> 8, (kMaxRun - since) >> 8);
      if (steps < kMinSteps || done) {
        if (distinct) flush();
        if (done) break;
        if (pend) idx = agg_home<SLOTS>((uint32_t)(word & kmask), (uint32_t)((word & kmask) >> 32));
        steps = kMaxSteps;
      }
      steps = min(steps, kMaxSteps);
      uint32_t acc = 0;  // new keys | windows merged << 12
      for (uint32_t st = 0; st < steps; st++) {
        if (!pend && rem) {
          if (left == 0) {
            cw = nxt;
            cm = nm;
            left = 32;
            nxt = rv.codes[wb + wnext];
            nm = rv.nmask[wb + wnext];
            wnext++;
          }
          const uint32_t b = (uint32_t)(cw >> 62);
          if (KHI) {
            const uint32_t fl = (uint32_t)fwd, fh = (uint32_t)(fwd >> 32);
            const uint32_t rl = (uint32_t)rcm, rh = (uint32_t)(rcm >> 32);
            fwd = ((uint64_t)(__builtin_amdgcn_alignbit(fh, fl, 30) & mhi) << 32) | ((fl << 2) | b);
            rcm = ((uint64_t)((rh >> 2) | ((b ^ 3u) << (rsh - 32))) << 32) | __builtin_amdgcn_alignbit(rh, rl, 2);
          } else {
            fwd = ((fwd << 2) | b) & kmask;
            rcm = (rcm >> 2) | ((uint64_t)(b ^ 3u) << rsh);
          }
          run = (int32_t)cm < 0 ? 0u : run + 1;
          cw <<= 2;
          cm <<= 1;
          left--;
          rem--;
          pend = run >= (uint32_t)k;
          take();
        }
        bool isnew = false, isin = false;
        if (pend) {
          const uint64_t old = atomicCAS((unsigned long long*)&s_tab[idx], 0ull, (unsigned long long)word);
          isnew = old == 0;
          const bool same = KHI ? ((uint32_t)old == (uint32_t)word &&
                                   (((uint32_t)(old >> 32) ^ (uint32_t)(word >> 32)) & khi) == 0)
                                : ((old ^ word) & t.kmo) == 0;
          if (same) atomicAdd((unsigned long long*)&s_tab[idx], (unsigned long long)one);
          isin = isnew || same;
          idx += agg_stride((uint32_t)word);
          idx = min(idx, idx - SLOTS);  // wraps: the difference is huge below SLOTS
          pend = !isin;
        }
        acc += (uint32_t)__popcll(__ballot(isnew)) + ((uint32_t)__popcll(__ballot(isin)) << 12);
        if (!__ballot(pend || rem)) break;
      }
      const uint64_t busy = __ballot(pend || rem);
      if (lane == 0) atomicAdd(&s_round[par], acc | (busy ? 1u << 24 : 0u));
      __syncthreads();
      const uint32_t v = __builtin_amdgcn_readfirstlane(s_round[par]);
      // the sums of the round after next: read by all before the last barrier, added to after the next
      par = par == 2 ? 0 : par + 1;
      if (tid == 0) s_round[par == 2 ? 0 : par + 1] = 0;
      distinct += v & 0xFFFu;
      since += (v >> 12) & 0xFFFu;
      if (EMIT && stage == 0) {
        stage = 1;
        if (nhave) {
          nL = rv.len[nr_];
          nwb = rv.word_off[nr_];
        }
      }
      done = !(v >> 24);
      if (done && !last) break;
    }
    L = nL;
    wb = nwb;
  }
  if (EMIT) {
    const uint64_t lim = cend < cap ? cend : cap;
    for (uint64_t i = cur + lane; i < lim; i += 64) out[i] = 0;
  }
  mynew = wave_sum_u32(mynew);
  if (lane == 0 && mynew) atomicAdd(&s_new, mynew);
  __syncthreads();
  if (tid == 0 && s_new)
    atomicAdd(reinterpret_cast<unsigned long long*>(&flags[2]), (unsigned long long)s_new);
}

// Groups of kReadsPerBlock consecutive positions of [r_begin, r_end), one table.
struct RangeGroups {
  uint64_t r_begin, r_end;
  __device__ __forceinline__ uint64_t count() const { return (r_end - r_begin + kReadsPerBlock - 1) / kReadsPerBlock; }
  __device__ __forceinline__ void get(uint64_t g, uint64_t& r0, int& nr, TableView&) const {
    r0 = r_begin + g * kReadsPerBlock;
    nr = (int)std::min<uint64_t>(kReadsPerBlock, r_end - r0);
  }
};

template <int SLOTS, bool EMIT, bool KHI>
__global__ __launch_bounds__(256, EMIT ? 5 : 4) void k_count_agg(
    ReadsView rv, uint64_t r_begin, uint64_t r_end, int k, int canonical, TableView t, uint32_t* __restrict__ flags,
    uint64_t* __restrict__ out, uint64_t cap, uint64_t chunk, unsigned long long* __restrict__ cursor,
    int table_ok) {
  count_agg<SLOTS, EMIT, KHI>(rv, RangeGroups{r_begin, r_end}, k, canonical, t, flags, out, cap, chunk, cursor,
                              table_ok);
}

}  // namespace tk
