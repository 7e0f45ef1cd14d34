// tk_iworm.hip -- Inchworm greedy contig construction over a count table.
//
// Replaces the assembly step of `inchworm --kmers <dump> --run_inchworm -K 25
// -L 25 --DS` (Trinity:2654-2711): seeds in order of count (descending, then
// key), each extended to the right and then to the left by the most abundant
// unused k-mer that overlaps the contig end by k-1 bases (ties: A<C<G<T),
// every k-mer used at most once.  The result is the serial greedy's, bit for
// bit, computed by many walks at once:
//
//  * seeds: the table's keys with count >= min_seed_cov (and a seed-entropy
//    composition table) sorted by key, then stably by inverted count;
//  * epochs: the next B seeds still unused are walked at once, sixteen
//    lanes per walk (four look up the candidate ending, or starting, with a
//    base).  Walk w of epoch base S has rank S+1+w; a walk claims each
//    k-mer it takes with atomicMin(claim[slot], rank), so a k-mer goes to the
//    earliest walk that wants it and a later walk that held it is marked lost.
//    A walk treats k-mers claimed by earlier ranks (committed epochs, or
//    earlier walks of this one) as used and records the latter;
//  * rounds: a walk holds if it lost no k-mer and every earlier walk whose
//    k-mers it treated as used holds and gives a contig, or if its seed was
//    taken by such a walk (skipped).  The others give their claims back and
//    are walked again with their ranks, the rest keep theirs, until all hold:
//    a round lasts as long as its longest walk, and few walks are ever in
//    conflict (3 to 16 of 16,384 beyond the seeds taken).  The earliest walk
//    of a round sees only walks that stay and so holds afterwards;
//  * commit: when every walk of the epoch holds, each equals the serial greedy
//    walk: the earlier walks it saw as claimers have exactly those k-mers, and
//    any k-mer an earlier serial walk takes was taken from it (it would be
//    lost).
//
// Claims are one u32 per table slot (tables of < 2^32 slots).
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <string>
#include <vector>

#include "tk_internal.h"

struct tk_contigs {
  int k = 25;
  std::string seq;
  std::vector<uint64_t> off{0};
  std::vector<uint64_t> sums;
  std::vector<uint64_t> seeds;
  uint64_t rounds = 0;
  uint64_t walks = 0;   // walks launched (committed or not)
  uint64_t steps = 0;   // k-mers appended by committed walks
};

namespace tk {

namespace {

constexpr uint32_t kFree = 0xFFFFFFFFu;
enum : uint32_t { kRunning = 0, kDone = 1, kSkip = 2, kLost = 3, kOverflow = 4 };

#define IW_LAUNCH(ctx, name, grid, block, kernel, ...)                                         \
  do {                                                                                         \
    hipEvent_t _a;                                                                             \
    ::tk::timing_begin((ctx), &_a);                                                            \
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), 0, (ctx)->stream, __VA_ARGS__);        \
    ::tk::timing_end((ctx), (name), _a);                                                       \
    hipError_t _le = hipGetLastError();                                                        \
    if (_le != hipSuccess) return ::tk::hip_fail(_le, "launch " name);                         \
  } while (0)

inline uint64_t cdiv(uint64_t a, uint64_t b) { return (a + b - 1) / b; }

// Count of key (0 when absent or pruned) and its global slot index (~0 when absent).
__device__ __forceinline__ uint64_t table_find(const TableView& t, uint64_t key, uint32_t* slot) {
  const uint64_t tagged = key | t.occ;
  uint64_t b = bucket0(t, key);
  for (uint32_t p = 0; p < t.max_probe; p++) {
    const ulonglong2* l2 = reinterpret_cast<const ulonglong2*>(t.slots + (b << 3));
    const ulonglong2 v0 = l2[0], v1 = l2[1], v2 = l2[2], v3 = l2[3];
    const uint64_t sv[8] = {v0.x, v0.y, v1.x, v1.y, v2.x, v2.y, v3.x, v3.y};
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const uint64_t s = sv[j];
      if ((s & t.kmo) == tagged) {
        *slot = (uint32_t)((b << 3) + j);
        return slot_count(t, s);
      }
      if (s == 0) {
        *slot = 0xFFFFFFFFu;
        return 0;
      }
    }
    b = bucket_next(t, b);
  }
  *slot = 0xFFFFFFFFu;
  return 0;
}

// Exchanges among a walk's sixteen lanes (a DPP row), by rotations of the row
// (one VALU instruction each; a shuffle goes through LDS).
template <int kRot>
__device__ __forceinline__ uint32_t row_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 + kRot, 0xF, 0xF, true);  // row_ror:kRot
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E;  // lanes 1032 and 2301 of four
template <int kPerm>
__device__ __forceinline__ uint32_t quad_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kPerm, 0xF, 0xF, true);
}
template <int kRot>
__device__ __forceinline__ uint64_t row_u64(uint64_t v) {
  return ((uint64_t)row_u32<kRot>((uint32_t)(v >> 32)) << 32) | row_u32<kRot>((uint32_t)v);
}
__device__ __forceinline__ uint64_t row_max_u64(uint64_t v) {
  v = std::max(v, row_u64<8>(v));
  v = std::max(v, row_u64<4>(v));
  v = std::max(v, row_u64<2>(v));
  return std::max(v, row_u64<1>(v));
}
// OR over the row: a value that one lane holds and the others pass 0 for.
__device__ __forceinline__ uint32_t row_or_u32(uint32_t v) {
  v |= row_u32<8>(v);
  v |= row_u32<4>(v);
  v |= row_u32<2>(v);
  return v | row_u32<1>(v);
}

// Seed candidates: (key, slot) of every slot with count >= min_cov whose
// composition passes keep (NULL: all), appended at *cursor (120 k reads' table:
// 1,009 -> 27 us with one atomic per tile instead of per wavefront).
__global__ __launch_bounds__(kScanThreads) void k_iw_seeds(TableView t, uint64_t n_slots, int k, uint64_t min_cov,
                                                           const uint8_t* __restrict__ keep,
                                                           uint64_t* __restrict__ keys, uint32_t* __restrict__ slots,
                                                           uint64_t cap, unsigned long long* __restrict__ cursor) {
  const uint64_t n2 = n_slots / 2;
  const uint64_t below = (1ull << (threadIdx.x & 63)) - 1;
  const int K1 = k + 1;
  for (uint64_t tile = blockIdx.x * kScanPairs; tile < n2; tile += gridDim.x * kScanPairs) {
    ulonglong2 v[kScanLoads];
    uint64_t m[2 * kScanLoads];
#pragma unroll
    for (int u = 0; u < kScanLoads; u++) v[u] = tile_pair(t.slots, tile, u, n2);
    uint32_t wtot = 0;
#pragma unroll
    for (int u = 0; u < 2 * kScanLoads; u++) {
      const uint64_t s = u & 1 ? v[u >> 1].y : v[u >> 1].x;
      bool take = false;
      if (s >> t.cshift) {
        const uint64_t n = slot_count(t, s);
        take = n >= min_cov && n > 0;
        if (take && keep) {
          int a, c, g;
          composition(s & (t.occ - 1), k, a, c, g);
          take = keep[(a * K1 + c) * K1 + g] != 0;
        }
      }
      m[u] = __ballot(take);
      wtot += (uint32_t)__popcll(m[u]);
    }
    uint64_t at = tile_reserve(wtot, cursor);
#pragma unroll
    for (int u = 0; u < 2 * kScanLoads; u++) {
      const uint64_t pos = at + (uint32_t)__popcll(m[u] & below);
      if (((m[u] >> (threadIdx.x & 63)) & 1ull) && pos < cap) {  // the host refuses a count past cap
        keys[pos] = (u & 1 ? v[u >> 1].y : v[u >> 1].x) & (t.occ - 1);
        slots[pos] = (uint32_t)(2 * (tile + (uint64_t)(u >> 1) * kScanThreads + threadIdx.x) + (u & 1));
      }
      at += (uint32_t)__popcll(m[u]);
    }
  }
}

// keys[i] = 2^32-1 - min(count of slot slots[i], 2^32-1): sorting by it
// (stably) orders seeds by count descending.
__global__ void k_iw_inv_count(TableView t, const uint32_t* __restrict__ slots, uint64_t n,
                               uint64_t* __restrict__ keys) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    uint64_t v = slot_count(t, t.slots[slots[i]]);
    v = v > 0xFFFFFFFFull ? 0xFFFFFFFFull : v;
    keys[i] = 0xFFFFFFFFull - v;
  }
}

__global__ void k_iw_fill(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// Committed claims keep their order only relative to new ranks: all become 1.
__global__ void k_iw_renumber(uint32_t* __restrict__ claim, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    if (claim[i] != kFree) claim[i] = 1u;
}

// One workgroup: the first `want` seeds from position `cursor` on whose slot
// is unclaimed.  out[0] = number picked; out64[1] = the position after the
// last one examined.  Each thread examines four consecutive positions per
// pass (their seed and claim loads in flight together), ranked by a block
// scan of the threads' counts, so a pass covers 4,096 positions.
constexpr uint32_t kPickPer = 4;

__global__ __launch_bounds__(1024) void k_iw_pick(const uint32_t* __restrict__ seeds, uint64_t n_seeds,
                                                  uint64_t cursor, const uint32_t* __restrict__ claim,
                                                  uint32_t want, uint32_t* __restrict__ picked_slot,
                                                  uint64_t* __restrict__ picked_pos,
                                                  unsigned long long* __restrict__ out) {
  __shared__ uint32_t s_wave[16];
  __shared__ uint32_t s_total;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t span = (uint64_t)kPickPer * blockDim.x;
  uint32_t got = 0;
  uint64_t base = cursor;
  uint64_t end = cursor;
  while (got < want && base < n_seeds) {
    const uint64_t p0 = base + (uint64_t)kPickPer * threadIdx.x;
    uint32_t sl[kPickPer];
    bool fr[kPickPer];
#pragma unroll
    for (uint32_t j = 0; j < kPickPer; j++) sl[j] = p0 + j < n_seeds ? seeds[p0 + j] : 0u;
    uint32_t cnt = 0;
#pragma unroll
    for (uint32_t j = 0; j < kPickPer; j++) {
      fr[j] = p0 + j < n_seeds && claim[sl[j]] == kFree;
      cnt += fr[j] ? 1u : 0u;
    }
    // inclusive scan of the counts within the wave, then across the waves
    uint32_t x = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o);
      if (lane >= o) x += y;
    }
    if (lane == 63) s_wave[wave] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t acc = 0;
      for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
        const uint32_t c = s_wave[w];
        s_wave[w] = acc;
        acc += c;
      }
      s_total = acc;
    }
    __syncthreads();
    uint32_t rank = got + s_wave[wave] + x - cnt;
#pragma unroll
    for (uint32_t j = 0; j < kPickPer; j++) {
      if (!fr[j]) continue;
      if (rank < want) {
        picked_slot[rank] = sl[j];
        picked_pos[rank] = p0 + j;
        if (rank == want - 1) out[1] = p0 + j + 1;  // the last picked seed ends the scan
      }
      rank++;
    }
    const uint32_t total = s_total;
    if (got + total >= want) {
      got = want;
    } else {
      got += total;
      end = std::min<uint64_t>(base + span, n_seeds);
    }
    base += span;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = got;
    if (got < want) out[1] = end;
  }
}

struct WalkParams {
  TableView t;
  uint64_t kmask;
  uint32_t S;       // ranks of this epoch: S+1 ... S+walks
  uint32_t n;       // walks of this round
  uint32_t lmax;    // path entries per walk and side
  int k;
  int canonical;
};

constexpr uint32_t kDeps = 8;  // recorded dependencies per walk (more: walked again as a round's first)

// Record that walk w treated a k-mer claimed by an earlier walk of this epoch
// (claim cl, the same on all lanes of the walk) as used: the decision holds
// only if that walk commits a contig.
__device__ __forceinline__ void iw_dep(uint32_t* __restrict__ deps, uint32_t* __restrict__ dep_n, uint32_t w,
                                       uint32_t S, uint32_t cl, uint32_t l16, uint32_t& last) {
  if (cl <= S || cl >= S + 1 + w || cl == last) return;
  last = cl;
  if (l16) return;
  const uint32_t j = dep_n[w];  // this lane alone counts them
  dep_n[w] = j + 1;
  if (j < kDeps) deps[w * kDeps + j] = cl - S - 1;
}

// Two slots of a candidate's home bucket and their claims, loaded but not yet
// looked at.
struct CandLoad {
  uint64_t tagged, b;
  ulonglong2 v;
  uint2 q;
};

// The k-mer after x on a side (0 right, all ones left) by base b, without a
// branch: a wait at its join would put the claim in flight before the loads.
__device__ __forceinline__ uint64_t iw_extend(const WalkParams& p, uint64_t x, uint64_t side, uint32_t b) {
  const uint64_t right = ((x << 2) | b) & p.kmask, left = ((uint64_t)b << (2 * (p.k - 1))) | (x >> 2);
  return right ^ ((right ^ left) & side);
}

__device__ __forceinline__ CandLoad iw_load(const WalkParams& p, const uint32_t* claim, uint64_t y, uint32_t part) {
  const uint64_t key = canon_key(y, p.k, p.canonical);
  CandLoad d;
  d.tagged = key | p.t.occ;
  d.b = bucket0(p.t, key);
  d.v = reinterpret_cast<const ulonglong2*>(p.t.slots + (d.b << 3))[part];
  d.q = reinterpret_cast<const uint2*>(claim + (d.b << 3))[part];
  return d;
}

// Count (0 = absent or pruned), slot and claim (possibly out of date) of a
// loaded candidate, on the lane of its four that holds it; 0 on the others.
__device__ __forceinline__ uint64_t iw_resolve(const TableView& t, const uint32_t* claim, const CandLoad& d,
                                               uint32_t part, uint32_t& slot, uint32_t& cl) {
  const bool m0 = (d.v.x & t.kmo) == d.tagged, m1 = (d.v.y & t.kmo) == d.tagged;
  slot = (uint32_t)(d.b << 3) + 2 * part + (m0 ? 0u : 1u);
  cl = m0 ? d.q.x : d.q.y;
  // full home bucket without it: the probe goes on, on the lane of its last slots
  const bool hit = m0 || m1;
  uint32_t any = hit ? 1u : 0u;
  any |= quad_u32<kQuadXor1>(any);
  any |= quad_u32<kQuadXor2>(any);
  uint64_t c = hit ? slot_count(t, m0 ? d.v.x : d.v.y) : 0;
  if (!any && part == 3 && d.v.y != 0) {
    c = table_find(t, d.tagged & (t.occ - 1), &slot);
    if (c) cl = claim[slot];
  }
  return c;
}

// Sixteen lanes per walk, four to a candidate base, two slots of its bucket to
// a lane: claim the seed, extend right, then left.  A walk is a chain of
// dependent steps and a round lasts as long as its longest walk, so the step's
// latency is what counts: a claim (a memory-side atomic), a lookup and the
// instructions between.  Claim and lookup run at once: the lookups of the step
// after are issued with the claim of the best candidate, as if it went
// through, and thrown away when it does not.  A candidate's claim word is
// loaded with its bucket, and one that an earlier rank is seen to hold is
// dropped without an atomic (claims only fall within a round, so what an
// out-of-date word says is held, is).  Each walk changes side on its own.
// 120 k reads' dictionary, 27 k steps: 3.98 -> 2.94 ms a round with the two at
// once, and 49.1 -> 43.8 ms in all from four lanes, each comparing the eight
// slots of a candidate, to sixteen.
__global__ __launch_bounds__(256) void k_iw_walk(WalkParams p, const uint32_t* __restrict__ list,
                                                 const uint32_t* __restrict__ picked_slot,
                                                 uint32_t* claim, uint32_t* __restrict__ lost,
                                                 uint32_t* __restrict__ status, uint32_t* __restrict__ lens,
                                                 uint64_t* __restrict__ sums, uint32_t* __restrict__ path_slot,
                                                 uint8_t* __restrict__ path_base, uint32_t* __restrict__ deps,
                                                 uint32_t* __restrict__ dep_n) {
  const uint32_t g = (blockIdx.x * blockDim.x + threadIdx.x) >> 4;
  if (g >= p.n) return;  // whole rows leave together
  const uint32_t w = list ? list[g] : g;
  const uint32_t l16 = threadIdx.x & 15, base = l16 >> 2, part = l16 & 3;
  const TableView& t = p.t;
  const uint32_t r = p.S + 1 + w;
  const uint32_t seed_slot = picked_slot[w];
  const uint64_t seed_word = t.slots[seed_slot];
  const uint64_t seed_key = seed_word & (t.occ - 1);
  uint64_t sum = slot_count(t, seed_word);
  uint32_t st = kRunning;
  uint32_t last_dep = 0;
  {
    uint32_t old = 0;
    if (l16 == 0) {
      old = atomicMin(&claim[seed_slot], r);
      if (old > r && old != kFree) atomicOr(&lost[old - p.S - 1], 1u);
    }
    old = row_or_u32(old);
    if (old < r) {
      st = kSkip;
      iw_dep(deps, dep_n, w, p.S, old, l16, last_dep);
    }
  }
  uint32_t nright = 0, len = 0;
  uint64_t side = 0;
  uint64_t x = seed_key;
  uint32_t* pslot = path_slot + (uint64_t)w * 2 * p.lmax;
  uint8_t* pbase = path_base + (uint64_t)w * 2 * p.lmax;
  if (st == kRunning) {
    uint32_t slot, cl;
    uint64_t c = iw_resolve(t, claim, iw_load(p, claim, iw_extend(p, x, side, base), part), part, slot, cl);
    for (;;) {
      // best remaining candidate: count, then smallest base; those seen held
      // by an earlier rank (or this walk) are dropped (c = 0)
      uint64_t best = 0;
      bool mine = false;
      for (;;) {
        const uint64_t my = c ? (((c < (1ull << 61) ? c : (1ull << 61)) << 2) | (3 - base)) : 0;
        best = row_max_u64(my);
        mine = my && my == best;
        const uint32_t held = row_or_u32(mine && cl <= r ? cl : 0u);
        if (!held) break;
        if (mine) c = 0;
        iw_dep(deps, dep_n, w, p.S, held, l16, last_dep);
      }
      if (best == 0) {  // this side ends here
        if (side) break;
        nright = len;
        side = ~0ull;
        len = 0;
        x = seed_key;
        pslot += p.lmax;
        pbase += p.lmax;
        c = iw_resolve(t, claim, iw_load(p, claim, iw_extend(p, x, side, base), part), part, slot, cl);
        continue;
      }
      if (len == p.lmax) {  // no room to record the claim: stop unclaimed
        st = kOverflow;
        break;
      }
      const uint32_t best_b = 3 - (uint32_t)(best & 3);
      uint32_t old = 0;
      if (mine) old = atomicMin(&claim[slot], r);
      // this walk's lost flag, the record (which does not count unless the
      // claim goes through) and the next step's lookups travel with the claim
      uint32_t l = 0;
      if (l16 == 0) l = __hip_atomic_load(&lost[w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (mine) {
        pslot[len] = slot;
        pbase[len] = (uint8_t)best_b;
      }
      const uint64_t xn = iw_extend(p, x, side, best_b);
      const CandLoad next = iw_load(p, claim, iw_extend(p, xn, side, base), part);
      old = row_or_u32(old);
      if (old <= r) {  // held by an earlier rank (or this walk)
        if (mine) c = 0;
        iw_dep(deps, dep_n, w, p.S, old, l16, last_dep);
        continue;
      }
      if (mine && old != kFree) atomicOr(&lost[old - p.S - 1], 1u);
      len++;
      // the count field of a taken slot is exact up to 2^61 (clamped above)
      sum += best >> 2;
      x = xn;
      if (row_or_u32(l)) {
        st = kLost;
        break;
      }
      c = iw_resolve(t, claim, next, part, slot, cl);
    }
    if (side == 0) nright = len, len = 0;
  }
  if (l16 == 0) {
    status[w] = st == kRunning ? kDone : st;
    lens[2 * w] = nright;
    lens[2 * w + 1] = len;
    sums[w] = sum;
  }
}

// Walks about to be walked again.
__global__ void k_iw_reset(const uint32_t* __restrict__ list, uint32_t n, uint32_t* __restrict__ lost,
                           uint32_t* __restrict__ dep_n) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    lost[list[i]] = 0;
    dep_n[list[i]] = 0;
  }
}

// The seed slot's claim of every walk (its own rank unless an earlier
// walk took the seed).
__global__ void k_iw_owner(const uint32_t* __restrict__ picked_slot, uint32_t n, const uint32_t* __restrict__ claim,
                           uint32_t* __restrict__ owner) {
  for (uint32_t w = blockIdx.x * blockDim.x + threadIdx.x; w < n; w += gridDim.x * blockDim.x)
    owner[w] = claim[picked_slot[w]];
}

// Flagged walks give their claims back (seed and path), a wave per walk (314 ->
// 13.5 us a round against a thread per side).
__global__ __launch_bounds__(256) void k_iw_release(uint32_t n, uint32_t S, uint32_t lmax,
                                                    const uint32_t* __restrict__ picked_slot,
                                                    const uint32_t* __restrict__ release,
                                                    const uint32_t* __restrict__ lens,
                                                    const uint32_t* __restrict__ path_slot,
                                                    uint32_t* __restrict__ claim) {
  const uint32_t lane = threadIdx.x & 63;
  for (uint32_t w = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; w < n; w += (gridDim.x * blockDim.x) >> 6) {
    if (!release[w]) continue;
    const uint32_t r = S + 1 + w;
    if (lane == 0) atomicCAS(&claim[picked_slot[w]], r, kFree);
#pragma unroll
    for (int side = 0; side < 2; side++) {
      const uint32_t* ps = path_slot + ((uint64_t)w * 2 + side) * lmax;
      const uint32_t len = lens[2 * w + side];
      for (uint32_t j = lane; j < len; j += 64) atomicCAS(&claim[ps[j]], r, kFree);
    }
  }
}

// One block per committed contig: left bases reversed, the seed, right bases.
__global__ __launch_bounds__(256) void k_iw_emit(const uint32_t* __restrict__ walks, const uint64_t* __restrict__ out_off,
                                                 const uint32_t* __restrict__ picked_slot, TableView t, int k,
                                                 uint32_t lmax, const uint32_t* __restrict__ lens,
                                                 const uint8_t* __restrict__ path_base, char* __restrict__ out) {
  const uint32_t w = walks[blockIdx.x];
  const uint32_t nr = lens[2 * w], nl = lens[2 * w + 1];
  const uint64_t key = t.slots[picked_slot[w]] & (t.occ - 1);
  const uint8_t* pr = path_base + ((uint64_t)w * 2) * lmax;
  const uint8_t* pl = path_base + ((uint64_t)w * 2 + 1) * lmax;
  char* o = out + out_off[blockIdx.x];
  const uint64_t L = (uint64_t)nl + k + nr;
  for (uint64_t i = threadIdx.x; i < L; i += blockDim.x) {
    uint32_t code;
    if (i < nl) code = pl[nl - 1 - i];
    else if (i < (uint64_t)nl + k) code = (uint32_t)((key >> (2 * (k - 1 - (i - nl)))) & 3);
    else code = pr[i - nl - k];
    o[i] = "ACGT"[code];
  }
}

struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  ~DevBuf() {
    if (p) dev_free(p, bytes);
  }
  int alloc(size_t b) {
    if (p) dev_free(p, bytes);
    p = nullptr;
    bytes = b;
    return dev_alloc(&p, b ? b : 8);
  }
  template <typename T>
  T* as() const {
    return (T*)p;
  }
};

int inchworm_run(tk_ctx* c, tk_table* t, uint32_t min_seed_cov, const uint8_t* seed_keep, tk_contigs* res) {
  const uint64_t n_slots = t->nb * 8;
  if (n_slots >= 0xFFFFFFFFull)
    return fail(TK_ERR_ARG, "inchworm: tables of 2^32 or more slots are not supported (%llu slots)",
                (unsigned long long)n_slots);
  const int k = t->k;
  TableView v = table_view(t);
  int rc;
  // ---- seeds in order: key ascending, then (stably) count descending
  DevBuf dkeep, dseedk, dseeds, dclaim;
  const int K1 = k + 1;
  if (seed_keep) {
    if ((rc = dkeep.alloc((size_t)K1 * K1 * K1))) return rc;
    TK_HIP(hipMemcpyAsync(dkeep.p, seed_keep, (size_t)K1 * K1 * K1, hipMemcpyHostToDevice, c->stream));
  }
  uint64_t n_cand = 0;
  {
    unsigned long long* cur = reinterpret_cast<unsigned long long*>(c->d_flags + 8);
    TK_HIP(hipMemsetAsync(cur, 0, 8, c->stream));
    // upper bound on seeds: the table's keys
    const uint64_t cap = std::max<uint64_t>(t->n_keys, 1);
    if ((rc = dseedk.alloc(cap * 8)) || (rc = dseeds.alloc(cap * 4))) return rc;
    IW_LAUNCH(c, "iworm_seeds", scan_grid(c, n_slots), kScanThreads, k_iw_seeds, v, n_slots, k,
              (uint64_t)min_seed_cov, seed_keep ? dkeep.as<uint8_t>() : nullptr, dseedk.as<uint64_t>(),
              dseeds.as<uint32_t>(), cap, cur);
    TK_HIP(hipMemcpyAsync(&n_cand, cur, 8, hipMemcpyDeviceToHost, c->stream));
    TK_HIP(hipStreamSynchronize(c->stream));
    if (n_cand > cap) return fail(TK_ERR_STATE, "inchworm: %llu seeds in a table of %llu keys",
                                  (unsigned long long)n_cand, (unsigned long long)cap);
    if ((rc = sort_pairs_u64_u32(c, dseedk.as<uint64_t>(), dseeds.as<uint32_t>(), n_cand, 2 * k))) return rc;
    if (n_cand)
      IW_LAUNCH(c, "iworm_order", std::min<uint64_t>(cdiv(n_cand, 256), 65536), 256, k_iw_inv_count, v,
                dseeds.as<uint32_t>(), n_cand, dseedk.as<uint64_t>());
    if ((rc = sort_pairs_u64_u32(c, dseedk.as<uint64_t>(), dseeds.as<uint32_t>(), n_cand, 32))) return rc;
  }
  if ((rc = dclaim.alloc(n_slots * 4))) return rc;
  IW_LAUNCH(c, "iworm_fill", std::min<uint64_t>(cdiv(n_slots, 256), 65536), 256, k_iw_fill,
            dclaim.as<uint32_t>(), n_slots, kFree);
  // ---- rounds
  // TK_IWORM_WALKS caps the walks per epoch (default 16,384, starting at
  // 1,024) and TK_IWORM_LMAX sets the first path capacity per walk side
  // (default 8,192 k-mers, 1.3 GB for a full epoch; 4,096 had 120 k reads' longest
  // contigs walked twice, 4 of 57 ms): small values force the conflict and regrowth
  // paths on small inputs.
  uint32_t Bmax = 16384, lmax = 8192;
  if (const char* e = getenv("TK_IWORM_WALKS")) Bmax = (uint32_t)std::min<unsigned long>(std::max(1ul, strtoul(e, nullptr, 10)), 16384ul);
  if (const char* e = getenv("TK_IWORM_LMAX")) lmax = (uint32_t)std::min<unsigned long>(std::max(4ul, strtoul(e, nullptr, 10)), 1ul << 20);
  const uint32_t Bmin = std::min<uint32_t>(64, Bmax);
  // path buffers hold Bcap walks: at most 2^28 path entries in all
  auto cap_for = [&](uint32_t lm) {
    return std::max<uint32_t>(Bmin, (uint32_t)std::min<uint64_t>(Bmax, (1ull << 28) / lm));
  };
  uint32_t Bcap = cap_for(lmax);
  uint32_t B = std::min<uint32_t>(1024, Bcap);
  DevBuf dpick, dpos, dout, dlost, dstat, dlens, dsums, dpslot, dpbase, dwalks, dwoff, dchars, ddeps, ddepn,
      downer, drel;
  if ((rc = dpick.alloc(Bmax * 4)) || (rc = dpos.alloc(Bmax * 8)) || (rc = dout.alloc(16)) ||
      (rc = dlost.alloc(Bmax * 4)) || (rc = dstat.alloc(Bmax * 4)) || (rc = dlens.alloc(Bmax * 8)) ||
      (rc = dsums.alloc(Bmax * 8)) || (rc = dwalks.alloc(Bmax * 4)) || (rc = dwoff.alloc(Bmax * 8 + 8)) ||
      (rc = ddeps.alloc((size_t)Bmax * kDeps * 4)) || (rc = ddepn.alloc(Bmax * 4)) || (rc = downer.alloc(Bmax * 4)) ||
      (rc = drel.alloc(Bmax * 4)))
    return rc;
  auto alloc_paths = [&]() -> int {
    int r2 = dpslot.alloc((size_t)Bcap * 2 * lmax * 4);
    if (!r2) r2 = dpbase.alloc((size_t)Bcap * 2 * lmax);
    return r2;
  };
  if (alloc_paths()) {  // no room for those: the smaller ones
    lmax = std::min(lmax, 4096u);
    if ((rc = alloc_paths())) return rc;
  }
  // the per-round host copies live in page-locked memory, so each is one DMA
  // (copies to pageable memory are staged and wait on the host)
  struct Pinned {
    void* p = nullptr;
    ~Pinned() {
      if (p) (void)hipHostFree(p);
    }
  } pin;
  // u32: stat, lost, lens (2), depn, owner, rel, walks, deps (kDeps) per walk;
  // u64: sums, pos, woff per walk, woff's end, out (2)
  const size_t u32s = (size_t)Bmax * (8 + kDeps), u64s = (size_t)Bmax * 3 + 1 + 2;
  TK_HIP(hipHostMalloc(&pin.p, u64s * 8 + u32s * 4, hipHostMallocDefault));
  uint64_t* h_sums = static_cast<uint64_t*>(pin.p);
  uint64_t* h_pos = h_sums + Bmax;
  uint64_t* h_woff = h_pos + Bmax;  // Bmax + 1
  unsigned long long* h_out = reinterpret_cast<unsigned long long*>(h_woff + Bmax + 1);  // 2
  uint32_t* h_stat = reinterpret_cast<uint32_t*>(h_out + 2);
  uint32_t* h_lost = h_stat + Bmax;
  uint32_t* h_lens = h_lost + Bmax;  // 2 * Bmax
  uint32_t* h_depn = h_lens + 2 * (size_t)Bmax;
  uint32_t* h_owner = h_depn + Bmax;
  uint32_t* h_rel = h_owner + Bmax;
  uint32_t* h_walks = h_rel + Bmax;
  uint32_t* h_deps = h_walks + Bmax;  // Bmax * kDeps
  enum : uint8_t { kBad, kContig, kSkipped };
  std::vector<uint8_t> state(Bmax), late(Bmax);  // late: its seed was taken by walk late_by while it ran
  std::vector<uint32_t> late_by(Bmax);
  uint64_t cursor = 0;
  uint32_t S = 0;
  std::string chunk;
  for (;;) {
    if ((uint64_t)S + 2ull * Bmax + 2 >= kFree) {
      IW_LAUNCH(c, "iworm_renumber", std::min<uint64_t>(cdiv(n_slots, 256), 65536), 256, k_iw_renumber,
                dclaim.as<uint32_t>(), n_slots);
      S = 1;
    }
    h_out[0] = h_out[1] = 0;
    IW_LAUNCH(c, "iworm_pick", 1, 1024, k_iw_pick, dseeds.as<uint32_t>(), n_cand, cursor, dclaim.as<uint32_t>(), B,
              dpick.as<uint32_t>(), dpos.as<uint64_t>(), dout.as<unsigned long long>());
    TK_HIP(hipMemcpyAsync(h_out, dout.p, 16, hipMemcpyDeviceToHost, c->stream));
    TK_HIP(hipStreamSynchronize(c->stream));
    const uint32_t n = (uint32_t)h_out[0];
    if (n == 0) break;
    IW_LAUNCH(c, "iworm_fill", cdiv(n, 256), 256, k_iw_fill, dlost.as<uint32_t>(), (uint64_t)n, 0u);
    IW_LAUNCH(c, "iworm_fill", cdiv(n, 256), 256, k_iw_fill, ddepn.as<uint32_t>(), (uint64_t)n, 0u);
    TK_HIP(hipMemcpyAsync(h_pos, dpos.p, (size_t)n * 8, hipMemcpyDeviceToHost, c->stream));
    WalkParams wp;
    wp.t = v;
    wp.kmask = k >= 32 ? ~0ull : ((1ull << (2 * k)) - 1);
    wp.S = S;
    wp.lmax = lmax;
    wp.k = k;
    wp.canonical = t->canonical;
    std::fill(late.begin(), late.begin() + n, 0);
    uint32_t m = n;         // walks of this round: all of the epoch, then h_walks[0 ... m)
    uint32_t first = 0;     // the earliest of them: it saw only walks that hold
    uint32_t P = n;         // committed walks
    bool outgrown = false;  // walk P outgrew its path buffers
    for (;;) {
      res->rounds++;
      res->walks += m;
      wp.n = m;
      IW_LAUNCH(c, "iworm_walk", cdiv((uint64_t)m * 16, 256), 256, k_iw_walk, wp,
                m == n ? nullptr : dwalks.as<uint32_t>(), dpick.as<uint32_t>(), dclaim.as<uint32_t>(),
                dlost.as<uint32_t>(), dstat.as<uint32_t>(), dlens.as<uint32_t>(), dsums.as<uint64_t>(),
                dpslot.as<uint32_t>(), dpbase.as<uint8_t>(), ddeps.as<uint32_t>(), ddepn.as<uint32_t>());
      IW_LAUNCH(c, "iworm_owner", cdiv(n, 256), 256, k_iw_owner, dpick.as<uint32_t>(), n, dclaim.as<uint32_t>(),
                downer.as<uint32_t>());
      TK_HIP(hipMemcpyAsync(h_depn, ddepn.p, n * 4, hipMemcpyDeviceToHost, c->stream));
      TK_HIP(hipMemcpyAsync(h_deps, ddeps.p, (size_t)n * kDeps * 4, hipMemcpyDeviceToHost, c->stream));
      TK_HIP(hipMemcpyAsync(h_owner, downer.p, n * 4, hipMemcpyDeviceToHost, c->stream));
      TK_HIP(hipMemcpyAsync(h_stat, dstat.p, n * 4, hipMemcpyDeviceToHost, c->stream));
      TK_HIP(hipMemcpyAsync(h_lost, dlost.p, n * 4, hipMemcpyDeviceToHost, c->stream));
      TK_HIP(hipMemcpyAsync(h_lens, dlens.p, (size_t)n * 8, hipMemcpyDeviceToHost, c->stream));
      TK_HIP(hipMemcpyAsync(h_sums, dsums.p, (size_t)n * 8, hipMemcpyDeviceToHost, c->stream));
      TK_HIP(hipStreamSynchronize(c->stream));
      // Which walks hold, in rank order.  A walk whose seed an earlier walk
      // took while it ran ("late") is the serial skip of that seed when the
      // taker gives a contig; its own claims are void.  Any decision that
      // treated a k-mer as used because an earlier walk held it (the
      // dependencies), and a seed found claimed at the start, holds only if
      // that walk gives a contig, i.e. is neither late nor skipped.  A walk
      // with more dependencies than are recorded holds if no earlier walk
      // changed since it started.
      uint32_t n_bad = 0;
      bool any_rel = false, full = false;  // full: the earliest walk that does not hold only lacked room
      for (uint32_t i = 0; i < n; i++) {
        const uint32_t r = S + 1 + i;
        auto contig = [&](uint32_t d) { return d < i && state[d] == kContig; };
        bool deps_ok = h_depn[i] <= kDeps || i <= first;  // those up to `first` have seen their last change
        for (uint32_t j = 0; deps_ok && j < std::min(h_depn[i], kDeps); j++)
          deps_ok = contig(h_deps[(size_t)i * kDeps + j]);
        h_rel[i] = 0;
        if (late[i]) {
          late[i] = contig(late_by[i]);
          state[i] = late[i] ? kSkipped : kBad;
        } else if (h_stat[i] == kSkip) {
          state[i] = deps_ok ? kSkipped : kBad;
        } else if (h_owner[i] != r) {  // seed taken by walk h_owner[i] - S - 1 < i
          late[i] = h_owner[i] > S && contig(h_owner[i] - S - 1);
          late_by[i] = h_owner[i] - S - 1;
          state[i] = late[i] ? kSkipped : kBad;
          h_rel[i] = late[i];
        } else {
          state[i] = h_stat[i] == kDone && !h_lost[i] && deps_ok ? kContig : kBad;
        }
        if (state[i] == kBad) {
          full = n_bad ? full : h_stat[i] == kOverflow && h_owner[i] == r && !h_lost[i] && deps_ok;
          h_rel[i] = 1;
          h_walks[n_bad++] = i;
        }
        any_rel = any_rel || h_rel[i];
      }
      if (n_bad && full) {
        // the earliest walk still open outgrew its path buffers: those before
        // it are committed, the rest is walked again with larger ones
        P = h_walks[0];
        outgrown = true;
        for (uint32_t i = P; i < n; i++) h_rel[i] = 1;
        any_rel = true;
      } else if (n_bad && h_walks[0] <= first) {
        return fail(TK_ERR_STATE, "inchworm: first walk of a round did not hold");
      }
      if (any_rel) {
        TK_HIP(hipMemcpyAsync(drel.p, h_rel, n * 4, hipMemcpyHostToDevice, c->stream));
        IW_LAUNCH(c, "iworm_release", cdiv((uint64_t)n * 64, 256), 256, k_iw_release, n, S,
                  lmax, dpick.as<uint32_t>(), drel.as<uint32_t>(), dlens.as<uint32_t>(), dpslot.as<uint32_t>(),
                  dclaim.as<uint32_t>());
      }
      if (!n_bad || outgrown) break;
      m = n_bad;
      first = h_walks[0];
      TK_HIP(hipMemcpyAsync(dwalks.p, h_walks, (size_t)m * 4, hipMemcpyHostToDevice, c->stream));
      IW_LAUNCH(c, "iworm_fill", cdiv(m, 256), 256, k_iw_reset, dwalks.as<uint32_t>(), m, dlost.as<uint32_t>(),
                ddepn.as<uint32_t>());
    }
    // contigs of the committed walks, in rank order
    uint32_t nw = 0;
    uint64_t total = 0;
    for (uint32_t i = 0; i < P; i++) {
      if (state[i] != kContig) continue;
      h_walks[nw] = i;
      h_woff[nw] = total;
      const uint64_t L = (uint64_t)h_lens[2 * i] + h_lens[2 * i + 1] + k;
      total += L;
      res->sums.push_back(h_sums[i]);
      res->seeds.push_back(0);  // filled from the sequence below
      res->steps += L - k;
      nw++;
    }
    if (nw) {
      if (dchars.bytes < total && (rc = dchars.alloc(std::max<uint64_t>(total, 1 << 20)))) return rc;
      TK_HIP(hipMemcpyAsync(dwalks.p, h_walks, (size_t)nw * 4, hipMemcpyHostToDevice, c->stream));
      TK_HIP(hipMemcpyAsync(dwoff.p, h_woff, (size_t)nw * 8, hipMemcpyHostToDevice, c->stream));
      IW_LAUNCH(c, "iworm_emit", nw, 256, k_iw_emit, dwalks.as<uint32_t>(), dwoff.as<uint64_t>(),
                dpick.as<uint32_t>(), v, k, lmax, dlens.as<uint32_t>(), dpbase.as<uint8_t>(), dchars.as<char>());
      chunk.resize(total);
      TK_HIP(hipMemcpyAsync(&chunk[0], dchars.p, total, hipMemcpyDeviceToHost, c->stream));
      TK_HIP(hipStreamSynchronize(c->stream));
      const uint64_t base_n = res->off.size() - 1;
      for (uint32_t j = 0; j < nw; j++) {
        const uint32_t i = h_walks[j];
        const uint64_t L = (uint64_t)h_lens[2 * i] + h_lens[2 * i + 1] + k;
        // seed key: the k bases after the left extension
        uint64_t key = 0;
        const char* s = chunk.data() + h_woff[j] + h_lens[2 * i + 1];
        for (int q = 0; q < k; q++) key = (key << 2) | (uint64_t)(s[q] == 'A' ? 0 : s[q] == 'C' ? 1 : s[q] == 'G' ? 2 : 3);
        res->seeds[base_n + j] = key;
        res->off.push_back(res->off.back() + L);
      }
      res->seq += chunk;
    }
    cursor = P < n ? h_pos[P] : h_out[1];
    S += n;
    if (!outgrown) {
      B = std::min(Bcap, B * 2);
      continue;
    }
    if (lmax >= (1u << 28)) return fail(TK_ERR_STATE, "inchworm: walk longer than 2^28 k-mers");
    TK_HIP(hipStreamSynchronize(c->stream));
    lmax *= 2;
    Bcap = cap_for(lmax);
    B = std::min(B, Bcap);
    if ((rc = alloc_paths())) return rc;
  }
  return TK_OK;
}

}  // namespace

}  // namespace tk

extern "C" {

int tk_inchworm(tk_ctx* c, tk_table* t, uint32_t min_seed_cov, const uint8_t* seed_keep, tk_contigs** out) {
  using namespace tk;
  if (!c || !t || !out) return fail(TK_ERR_ARG, "NULL argument");
  *out = nullptr;
  if (hipSetDevice(c->device) != hipSuccess) return fail(TK_ERR_HIP, "hipSetDevice");
  int rc = table_finalize(c, t);
  if (rc) return rc;
  tk_contigs* r = new tk_contigs();
  r->k = t->k;
  rc = inchworm_run(c, t, min_seed_cov, seed_keep, r);
  (void)hipStreamSynchronize(c->stream);
  if (rc) {
    delete r;
    return rc;
  }
  *out = r;
  return TK_OK;
}

int tk_contigs_info(const tk_contigs* r, uint64_t* n_contigs, uint64_t* total_len, uint64_t* rounds,
                    uint64_t* walks) {
  if (!r) return tk::fail(TK_ERR_ARG, "NULL argument");
  if (n_contigs) *n_contigs = r->off.size() - 1;
  if (total_len) *total_len = r->seq.size();
  if (rounds) *rounds = r->rounds;
  if (walks) *walks = r->walks;
  return TK_OK;
}

int tk_contigs_get(const tk_contigs* r, char* seq, uint64_t* offsets, uint64_t* sums, uint64_t* seed_keys) {
  if (!r) return tk::fail(TK_ERR_ARG, "NULL argument");
  const size_t n = r->off.size() - 1;
  if (seq && !r->seq.empty()) memcpy(seq, r->seq.data(), r->seq.size());
  if (offsets) memcpy(offsets, r->off.data(), (n + 1) * 8);
  if (sums && n) memcpy(sums, r->sums.data(), n * 8);
  if (seed_keys && n) memcpy(seed_keys, r->seeds.data(), n * 8);
  return TK_OK;
}

int tk_contigs_free(tk_contigs* r) {
  delete r;
  return TK_OK;
}

}  // extern "C"
