// tk_device.h -- device-side building blocks shared by the gfx950 kernels.
//
// Read layout in HBM (tk_reads):
//   codes[w]  : 64-bit word, 32 bases, 2 bits each, first base in bits 63..62
//   nmask[w]  : 32-bit word, bit 31-i set when base i of codes[w] is not ACGT
//   word_off[r]: first word of read r (each read starts on a fresh word)
//   len[r]    : bases in read r
// kWordPad padding words (code 0, every base invalid) follow the last read, so
// a window extractor may always read words w and w+1, and a lane of a
// per-read kernel the four words from its own on (lane_words).
//
// Count table (tk_table): open addressing over 64-byte buckets of eight
// 64-bit slots.  A slot packs
//     [ count field : 63-2k bits | occupied : 1 bit | key : 2k bits ]
// so one 64-bit atomicAdd of (1 << (2k+1)) increments a k-mer and any carry
// leaves through bit 63 without touching the key.  A carry (field wrap) is
// recorded as 2^(63-2k) in a small side table keyed by k-mer ("ovf").
// Finalisation folds the side table back: the main field of every key with
// a side entry becomes all-ones and the side entry holds the full count.
// A field of 0 on an occupied, finalised slot is a pruned key (tombstone).
//
// Buckets are grouped into regions of 2^rbits consecutive buckets; the table
// holds nb = P * 2^rbits buckets.  A key's home bucket is
// mulhi(mix64(key), nb) and probing wraps inside the home region, so every
// key stays in one region.  Counting can then be done region by region with
// the active region resident in the Infinity Cache.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tk {

constexpr int kWave = 64;
constexpr int kBucketSlots = 8;
constexpr int kWordPad = 16;
// u64 entries of LDS lookup scratch per wavefront (coop_lookup: 64 two-word
// entries, then up to 128 values)
constexpr int kLookupScratch = 128;

__host__ __device__ __forceinline__ uint64_t mix64(uint64_t x) {
  x ^= x >> 33;
  x *= 0xff51afd7ed558ccdULL;
  x ^= x >> 33;
  x *= 0xc4ceb9fe1a85ec53ULL;
  x ^= x >> 33;
  return x;
}

// Reverse complement of a k-mer held in the low 2k bits: the bits reversed
// (bases reversed, the two bits of each swapped), the pairs swapped back.
__device__ __forceinline__ uint64_t revcomp(uint64_t v, int k) {
  const uint64_t x = __builtin_bitreverse64(~v);
  return (((x >> 1) & 0x5555555555555555ULL) | ((x & 0x5555555555555555ULL) << 1)) >> (64 - 2 * k);
}

struct ReadsView {
  const uint64_t* codes;
  const uint32_t* nmask;
  const uint64_t* word_off;
  const uint32_t* len;
  uint64_t n_reads;
  const uint32_t* order = nullptr;  // processing order of the table passes (nullptr = input order)
};

// Read processed at position i of the table passes.
__device__ __forceinline__ uint64_t read_at(const ReadsView& rv, uint64_t i) {
  return rv.order ? rv.order[i] : i;
}

// Workgroup b of a launch runs on XCD b % 8 (round-robin dispatch).  For a
// grid that is a multiple of 8 this maps b to a logical block such that each
// XCD takes one contiguous run of logical blocks, so work adjacent in the
// read order shares that XCD's L2.
__device__ __forceinline__ uint64_t xcd_block(uint64_t b, uint64_t grid) {
  return (b & 7) * (grid >> 3) + (b >> 3);
}

// Per-XCD position counters of the per-read table passes: eight u32, one per
// 256 B, cleared before each launch.
constexpr uint32_t kTicketStride = 64;
constexpr uint32_t kTicketWords = 8 * kTicketStride;

// Positions [0, n) of one XCD's share of a per-read pass, for one wave.
// kTicket: the XCD's waves take runs of `grab` consecutive positions from
// that XCD's counter *ctr (one returning atomic per run; the next run is
// taken while the current one is processed), so the positions in flight on
// the XCD stay one narrow front of the order however far single waves drift
// apart.  Otherwise the wave takes first, first + stride, ... (a fixed
// stride, along which waves drift apart by thousands of reads on large sets).
// Calls f(position) for each; every wave leaves once its next position is at
// or past n.
template <bool kTicket, class F>
__device__ __forceinline__ void xcd_positions(uint32_t* ctr, uint64_t n, uint32_t grab, uint64_t first,
                                              uint64_t stride, int lane, F&& f) {
  if (!kTicket) {
    for (uint64_t j = first; j < n; j += stride) f(j);
    return;
  }
  // positions fit 32 bits: a share is at most 2^31 / 8 reads
  const uint32_t n32 = (uint32_t)n;
  uint32_t t = 0;
  if (lane == 0) t = atomicAdd(ctr, grab);
  uint32_t b = __shfl(t, 0);
  while (b < n32) {
    t = 0;
    if (lane == 0) t = atomicAdd(ctr, grab);
    const uint32_t e = n32 - b > grab ? b + grab : n32;
    for (uint32_t j = b; j < e; j++) f(j);
    b = __shfl(t, 0);
  }
}

// The positions of xcd_positions<true>, one at a time: next() gives the
// wave's next position of [0, n), and n once the XCD's share is used up.
struct TicketStream {
  uint32_t* ctr;
  uint32_t n, grab;
  uint32_t cb = 0, ce = 0;  // current run [cb, ce)
  uint32_t tk = 0;          // lane 0: start of the run taken next
  bool done = false;
  int lane;
  __device__ __forceinline__ TicketStream(uint32_t* c, uint32_t n_, uint32_t g, int l)
      : ctr(c), n(n_), grab(g), lane(l) {
    if (lane == 0) tk = atomicAdd(ctr, grab);
  }
  __device__ __forceinline__ uint32_t next() {
    if (cb == ce) {
      if (done) return n;
      const uint32_t s = __builtin_amdgcn_readfirstlane(tk);
      if (s >= n) {
        done = true;
        return n;
      }
      cb = s;
      ce = n - s > grab ? s + grab : n;
      if (lane == 0) tk = atomicAdd(ctr, grab);
    }
    return cb++;
  }
};

// Forward k-mer starting at base `pos` of the read whose first word is wbase.
__device__ __forceinline__ void window_at(const ReadsView& rv, uint64_t wbase,
                                          uint32_t pos, int k, uint64_t& fwd,
                                          bool& valid) {
  const uint64_t w = wbase + (pos >> 5);
  const uint32_t o = pos & 31u;
  const uint64_t hi = rv.codes[w];
  const uint64_t lo = rv.codes[w + 1];
  const uint32_t mhi = rv.nmask[w];
  const uint32_t mlo = rv.nmask[w + 1];
  const uint64_t x = o ? ((hi << (2 * o)) | (lo >> (64 - 2 * o))) : hi;
  const uint32_t m = o ? ((mhi << o) | (mlo >> (32 - o))) : mhi;
  fwd = x >> (64 - 2 * k);
  valid = (m >> (32 - k)) == 0u;
}

// The words a lane needs for its two windows of a run of 128 (windows lane and
// 64 + lane of a read whose words start at wb): words lane/32 .. lane/32 + 3.
// Every lane loads its own (three 16-byte loads, one or two lines per wave),
// which replaced words spread over the lanes and fetched with six shuffles per
// window.  Words are 8-byte aligned, masks 4-byte: the vector types say so.
typedef uint64_t words2 __attribute__((ext_vector_type(2), aligned(8)));
typedef uint32_t masks4 __attribute__((ext_vector_type(4), aligned(4)));

struct LaneWords {
  words2 a, b;  // words 0-1 and 2-3
  masks4 m;
};

__device__ __forceinline__ LaneWords lane_words(const ReadsView& rv, uint64_t wb, int lane) {
  const uint32_t j = (uint32_t)lane >> 5;
  LaneWords w;
  w.a = *reinterpret_cast<const words2*>(rv.codes + wb + j);
  w.b = *reinterpret_cast<const words2*>(rv.codes + wb + j + 2);
  w.m = *reinterpret_cast<const masks4*>(rv.nmask + wb + j);
  return w;
}

// Last read whose first word is at or before word w (the read holding w; empty
// reads before it are passed over), found by the whole wave: 64 pivots a step.
__device__ __forceinline__ uint64_t read_of_word(const uint64_t* __restrict__ word_off, uint64_t n_reads, uint64_t w,
                                                 int lane) {
  uint64_t lo = 0, hi = n_reads;
  while (hi - lo > 1) {
    const uint64_t step = (hi - lo + 63) >> 6;
    const uint64_t p = lo + (uint64_t)lane * step;
    const uint64_t m = __ballot(p < hi && word_off[p] <= w);
    lo += (uint64_t)(63 - __clzll((long long)(m | 1ull))) * step;
    hi = hi < lo + step ? hi : lo + step;
  }
  return lo;
}

// The read holding word w, from a read r on whose first word is at or before
// it: r or one of the next few, or by bisection past a run of empty reads.
__device__ __forceinline__ uint64_t read_from(const uint64_t* __restrict__ word_off, uint64_t n_reads, uint64_t r,
                                              uint64_t w) {
  for (int i = 0; i < 4; i++) {
    if (word_off[r + 1] > w) return r;
    r++;
  }
  uint64_t hi = n_reads;
  while (hi - r > 1) {
    const uint64_t mid = r + ((hi - r) >> 1);
    if (word_off[mid] <= w) r = mid;
    else hi = mid;
  }
  return r;
}

// Forward k-mer at base o (< 32) of the word pair (hi, lo) with masks (mhi, mlo).
__device__ __forceinline__ void pair_window(uint64_t hi, uint64_t lo, uint32_t mhi, uint32_t mlo, uint32_t o, int k,
                                            uint64_t& fwd, bool& valid) {
  const uint64_t x = (hi << (2 * o)) | ((lo >> 1) >> (63 - 2 * o));
  const uint32_t m = (mhi << o) | ((mlo >> 1) >> (31 - o));
  fwd = x >> (64 - 2 * k);
  valid = (m >> (32 - k)) == 0u;
}

__device__ __forceinline__ uint64_t canon_key(uint64_t fwd, int k, int canonical) {
  if (!canonical) return fwd;
  const uint64_t rc = revcomp(fwd, k);
  return rc < fwd ? rc : fwd;
}

struct TableView {
  uint64_t* slots;    // base of the slot array (shared by the tables of a batch)
  uint64_t boff;      // first bucket of this table
  uint64_t nb;        // buckets
  uint64_t rmask;     // buckets per region - 1
  uint32_t rbits;     // log2(buckets per region)
  uint64_t occ;       // occupied bit (1 << 2k)
  uint64_t kmo;       // key + occupied bits
  uint64_t cmax;      // all-ones count field value
  uint32_t cshift;    // 2k + 1
  uint32_t cbits;     // 63 - 2k
  uint64_t* ovf;      // side table: pairs (tagged key, value)
  uint64_t omask;     // side capacity - 1
  uint32_t max_probe; // buckets probed before giving up
};

// High 64 bits of h * n.  n (a table's buckets) is the same for every lane
// and below 2^32 but for tables of 256 GB, so half of the product's four
// quarter-rate 32-bit multiplies go, behind a scalar branch.
__device__ __forceinline__ uint64_t mulhi_n(uint64_t h, uint64_t n) {
  if (n >> 32) return __umul64hi(h, n);
  const uint32_t n32 = (uint32_t)n;
  return ((uint64_t)(uint32_t)(h >> 32) * n32 + __umulhi((uint32_t)h, n32)) >> 32;
}

__device__ __forceinline__ uint64_t bucket0(const TableView& t, uint64_t key) {
  return t.boff + mulhi_n(mix64(key), t.nb);
}
__device__ __forceinline__ uint64_t bucket_next(const TableView& t, uint64_t b) {
  const uint64_t r = b - t.boff;
  return t.boff + ((r & ~t.rmask) | ((r + 1) & t.rmask));
}

// ---- side table (field carries) ----
__device__ __forceinline__ uint64_t ovf_slot0(const TableView& t, uint64_t tagged) {
  return mix64(tagged ^ 0x9E3779B97F4A7C15ULL) & t.omask;
}

__device__ inline void ovf_add(const TableView& t, uint64_t tagged, uint64_t units,
                               uint32_t* err) {
  uint64_t i = ovf_slot0(t, tagged);
  for (uint64_t p = 0; p <= t.omask; p++) {
    unsigned long long* kp = (unsigned long long*)&t.ovf[2 * i];
    uint64_t cur = *kp;
    if (cur == 0) {
      cur = atomicCAS(kp, 0ULL, (unsigned long long)tagged);
      if (cur == 0) cur = tagged;
    }
    if (cur == tagged) {
      atomicAdd((unsigned long long*)&t.ovf[2 * i + 1], (unsigned long long)units);
      return;
    }
    i = (i + 1) & t.omask;
  }
  atomicOr(err, 2u);
}

__device__ inline uint64_t* ovf_find(const TableView& t, uint64_t tagged) {
  uint64_t i = ovf_slot0(t, tagged);
  for (uint64_t p = 0; p <= t.omask; p++) {
    uint64_t cur = t.ovf[2 * i];
    if (cur == tagged) return &t.ovf[2 * i + 1];
    if (cur == 0) return nullptr;
    i = (i + 1) & t.omask;
  }
  return nullptr;
}

// Add r (< 2^cbits) to the count field of slot `s` and q (a multiple of
// 2^cbits) plus any carry to the side table.
__device__ __forceinline__ void field_add(const TableView& t, uint64_t* s, uint64_t tagged,
                                          uint64_t r, uint64_t q, uint32_t* err) {
  if (r) {
    const uint64_t old = atomicAdd((unsigned long long*)s, (unsigned long long)(r << t.cshift));
    if ((old >> t.cshift) + r > t.cmax) q += t.cmax + 1;
  }
  if (q) ovf_add(t, tagged, q, err);
}

// Insert-or-add c >= 1 occurrences of key.  Returns 1 when a new slot was
// claimed, 0 when the key was present, 2 when max_probe buckets were full
// (nothing added; the caller decides).
__device__ inline uint32_t table_add(const TableView& t, uint64_t key, uint64_t c,
                                     uint32_t* err) {
  const uint64_t tagged = key | t.occ;
  const uint64_t r = c & t.cmax;
  const uint64_t q = c - r;
  uint64_t b = bucket0(t, key);
  for (uint32_t p = 0; p < t.max_probe; p++) {
    uint64_t* line = t.slots + (b << 3);
    const ulonglong2* l2 = reinterpret_cast<const ulonglong2*>(line);
    ulonglong2 v0 = l2[0], v1 = l2[1], v2 = l2[2], v3 = l2[3];
    uint64_t sv[8] = {v0.x, v0.y, v1.x, v1.y, v2.x, v2.y, v3.x, v3.y};
#pragma unroll
    for (int j = 0; j < 8; j++) {
      uint64_t s = sv[j];
      if (s == 0) {
        s = atomicCAS((unsigned long long*)&line[j], 0ULL,
                      (unsigned long long)(tagged | (r << t.cshift)));
        if (s == 0) {
          if (q) ovf_add(t, tagged, q, err);
          return 1u;
        }
      }
      if ((s & t.kmo) == tagged) {
        field_add(t, &line[j], tagged, r, q, err);
        return 0u;
      }
    }
    b = bucket_next(t, b);
  }
  return 2u;
}

// Count of key in a finalised table; 0 when absent or pruned.
__device__ __forceinline__ uint64_t table_get(const TableView& t, uint64_t key) {
  const uint64_t tagged = key | t.occ;
  uint64_t b = bucket0(t, key);
  for (uint32_t p = 0; p < t.max_probe; p++) {
    const ulonglong2* l2 = reinterpret_cast<const ulonglong2*>(t.slots + (b << 3));
    ulonglong2 v0 = l2[0], v1 = l2[1], v2 = l2[2], v3 = l2[3];
    uint64_t sv[8] = {v0.x, v0.y, v1.x, v1.y, v2.x, v2.y, v3.x, v3.y};
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const uint64_t s = sv[j];
      if ((s & t.kmo) == tagged) {
        const uint64_t f = s >> t.cshift;
        if (f != t.cmax) return f;
        const uint64_t* o = ovf_find(t, tagged);
        return o ? *o : f;
      }
      if (s == 0) return 0;
    }
    b = bucket_next(t, b);
  }
  return 0;
}

// Count of the key held by an occupied slot value (finalised table).
__device__ __forceinline__ uint64_t slot_count(const TableView& t, uint64_t s) {
  const uint64_t f = s >> t.cshift;
  if (f != t.cmax) return f;
  const uint64_t* o = ovf_find(t, s & t.kmo);
  return o ? *o : f;
}

// ---- LDS tables with an 8-bit tag per slot ----
// Tag of a key from its mix64 hash (low byte; the bucket comes from the high
// bits): 1..255, 0 marks a slot with no tag yet.
__device__ __forceinline__ uint32_t slot_tag(uint64_t h) {
  const uint32_t t8 = (uint32_t)h & 0xFFu;
  return t8 ? t8 : 1u;
}

// 0x80 in every byte of x that is zero, 0 elsewhere (exact: no carries
// between bytes).
__device__ __forceinline__ uint64_t zero_bytes(uint64_t x) {
  const uint64_t m = 0x7F7F7F7F7F7F7F7Full;
  return ~(((x & m) + m) | x | m);
}

// Insert-or-add into an LDS table of nb buckets of eight 8-B slots in the
// global slot format, with tags[8 * b + j] the tag of slot j of bucket b:
// `word` = tagged key | c << cshift.  A step reads the bucket's eight tags (8
// bytes), reads only the slots whose tag matches (to confirm the key), and
// otherwise claims the first slot with no tag by CAS, then writes its tag.
// A slot claimed but not yet tagged by another thread shows as untagged: the
// CAS then fails, and the slot is taken as the key's (add) or skipped.
// Occupied slots stay a prefix of their bucket.  Returns 2 when a slot was
// claimed, 1 when added (old = previous slot value), 0 when max_steps steps
// found no room.
__device__ __forceinline__ int lds_tag_add(uint64_t* tab, uint8_t* tags, uint32_t b, uint32_t nb, uint64_t word,
                                           uint32_t tag, uint64_t kmo, uint32_t cshift, uint32_t max_steps,
                                           uint64_t& old) {
  const uint64_t tagged = word & kmo;
  const uint64_t add = (word >> cshift) << cshift;
  const uint64_t rep = 0x0101010101010101ull * tag;
  uint64_t skip = 0;  // bytes of slots known to hold other keys
  for (uint32_t p = 0; p < max_steps; p++) {
    uint64_t* line = tab + ((uint64_t)b << 3);
    const uint64_t tw = *reinterpret_cast<const uint64_t*>(tags + ((uint64_t)b << 3));
    const uint64_t em = zero_bytes(tw) & ~skip;
    uint64_t mm = zero_bytes(tw ^ rep) & ~skip;
    const uint32_t je = em ? (uint32_t)__builtin_ctzll(em) >> 3 : 8u;
    while (mm) {
      const uint32_t j = (uint32_t)__builtin_ctzll(mm) >> 3;
      if (j >= je) break;
      const uint64_t v = line[j];
      if ((v & kmo) == tagged) {
        old = atomicAdd((unsigned long long*)&line[j], (unsigned long long)add);
        return 1;
      }
      skip |= 0xFFull << (8 * j);
      mm &= mm - 1;
    }
    if (je < 8) {
      const uint64_t v = atomicCAS((unsigned long long*)&line[je], 0ull, (unsigned long long)word);
      if (v == 0) {
        tags[((uint64_t)b << 3) + je] = (uint8_t)tag;
        return 2;
      }
      if ((v & kmo) == tagged) {
        old = atomicAdd((unsigned long long*)&line[je], (unsigned long long)add);
        return 1;
      }
      skip |= 0xFFull << (8 * je);
      continue;  // rescan this bucket past the slot another key took
    }
    b = b + 1 == nb ? 0 : b + 1;
    skip = 0;
  }
  return 0;
}

// ---- wave helpers ----
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Bit g of the result is set when byte g of x is non-zero.
__device__ __forceinline__ uint32_t byte_any8(uint64_t x) {
  x |= x >> 4;
  x |= x >> 2;
  x |= x >> 1;
  x &= 0x0101010101010101ULL;
  return (uint32_t)((x * 0x0102040810204080ULL) >> 56);
}

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
// Adds the block's sum of v to *out with one atomic (every thread of the
// block must call it; blockDim <= 1024).  Atomics on one address are
// serialized at the memory side, so one per wavefront of a large grid costs
// milliseconds.
__device__ __forceinline__ void block_sum_add(uint64_t v, unsigned long long* out) {
  __shared__ uint64_t s_part[16];
  v = wave_sum_u64(v);
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t tot = 0;
    for (uint32_t w = 0; w < (blockDim.x + 63) / 64; w++) tot += s_part[w];
    if (tot) atomicAdd(out, (unsigned long long)tot);
  }
}
// Wave reductions of 32-bit values on the DPP row shifts and row broadcasts
// (one VALU instruction per step; a shuffle is an address, an LDS permute and
// a wait).  All 64 lanes must be active; the result is wave-uniform.
template <int kCtrl, int kRows>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t identity, uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)identity, (int)v, kCtrl, kRows, 0xF, false);
}
template <class Op>
__device__ __forceinline__ uint32_t wave_reduce_u32(uint32_t v, uint32_t identity, Op op) {
  v = op(v, dpp_u32<0x111, 0xF>(identity, v));  // row_shr:1
  v = op(v, dpp_u32<0x112, 0xF>(identity, v));  // row_shr:2
  v = op(v, dpp_u32<0x114, 0xF>(identity, v));  // row_shr:4
  v = op(v, dpp_u32<0x118, 0xF>(identity, v));  // row_shr:8: lane 15 of a row holds the row's result
  v = op(v, dpp_u32<0x142, 0xA>(identity, v));  // row_bcast:15 into rows 1 and 3
  v = op(v, dpp_u32<0x143, 0xC>(identity, v));  // row_bcast:31 into rows 2 and 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t v) {
  return wave_reduce_u32(v, 0u, [](uint32_t a, uint32_t b) { return a + b; });
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  return wave_reduce_u32(v, 0u, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
  return wave_reduce_u32(v, 0xFFFFFFFFu, [](uint32_t a, uint32_t b) { return a < b ? a : b; });
}

// ---- passes over the slots of a finished table ----
// The scans that append what they find (dump, Inchworm's seeds) take tiles of
// 4,096 slots per block of 512 threads, four 16-byte loads in flight per
// thread, and reserve a tile's output with one atomic on the cursor: with one
// per wavefront of 64 slots the memory side, which serializes atomics on one
// address (about 19 ns each), set the pace.  Grids are a few blocks per CU for
// the same reason (each block ends in at most one more atomic).
constexpr int kScanThreads = 512;
constexpr int kScanLoads = 4;  // ulonglong2 per thread and tile
constexpr uint64_t kScanPairs = (uint64_t)kScanThreads * kScanLoads;

// First output position of this wavefront's `wtot` items of the block's tile.
// Every thread of the block (kScanThreads) calls it.
__device__ __forceinline__ uint64_t tile_reserve(uint32_t wtot, unsigned long long* cursor) {
  __shared__ uint32_t s_w[kScanThreads / 64];
  __shared__ unsigned long long s_base;
  const int wv = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) s_w[wv] = wtot;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t tot = 0;
    for (int i = 0; i < kScanThreads / 64; i++) tot += s_w[i];
    s_base = tot ? atomicAdd(cursor, (unsigned long long)tot) : 0ull;
  }
  __syncthreads();
  uint64_t at = s_base;
  for (int i = 0; i < wv; i++) at += s_w[i];
  __syncthreads();  // s_w and s_base are read before the next tile writes them
  return at;
}

// Slot pair u of this thread in the tile at pair `tile` (zeros past the end).
__device__ __forceinline__ ulonglong2 tile_pair(const uint64_t* slots, uint64_t tile, int u, uint64_t n2) {
  const uint64_t i = tile + (uint64_t)u * kScanThreads + threadIdx.x;
  return i < n2 ? reinterpret_cast<const ulonglong2*>(slots)[i] : make_ulonglong2(0ull, 0ull);
}

// Numbers of A, C and G in a k-mer.
__device__ __forceinline__ void composition(uint64_t key, int k, int& a, int& c, int& g) {
  const uint64_t M = 0x5555555555555555ULL & ((1ull << (2 * k)) - 1);  // k <= 31
  const uint64_t lo = key & M, hi = (key >> 1) & M;
  const int nt = __popcll(hi & lo);
  g = __popcll(hi & ~lo & M);
  c = __popcll(~hi & lo & M);
  a = k - nt - g - c;
}

// Bit g of the result is set when nibble g (lanes 4g..4g+3) of x is non-zero.
__device__ __forceinline__ uint32_t nibble_bits(uint64_t x) {
  x |= x >> 1;
  x |= x >> 2;
  x &= 0x1111111111111111ULL;
  x = (x | (x >> 3)) & 0x0303030303030303ULL;
  x = (x | (x >> 6)) & 0x000F000F000F000FULL;
  x = (x | (x >> 12)) & 0x000000FF000000FFULL;
  return (uint32_t)((x | (x >> 24)) & 0xFFFFu);
}

// Cooperative lookup of 64*NK keys, NK per lane (key i of a lane is key
// number 64*i + lane), four lanes per key.  In round q the lanes 4g..4g+3
// read the 64-byte home bucket of key 16q+g, sixteen bytes each: one
// coalesced request per key.  All 4*NK loads of a lane are issued before any
// is inspected.
//
// The kernels that call this are bound by instruction issue as much as by
// their misses (the scoring pass issued vector instructions in 76% of its
// cycles), so the exchange between a key's lane and its group goes through
// LDS: the lane writes {bucket offset, tagged key} once and the group reads
// both with one broadcast 16-byte read per round (five shuffles before).  The
// matching lane writes the key's value back; a group whose bucket is full
// (its last lane sees no empty slot; occupied slots are a prefix) first
// leaves kLookupFull there, which a match overwrites (the LDS operations of a
// wave execute in order), and the key's lane then probes on alone.
//
// off[i]: byte offset of the home bucket from `slots`.  Layout L: match(slots,
// tag, value) for the lane's sixteen bytes, full(slots) for the bucket's last
// sixteen, kNone the value of an absent key.  A lane without a key asks for
// bucket 0 with tag 0 (no branch around the loads) and ignores its value.
// scratch: kLookupScratch u64.
constexpr uint64_t kLookupFull = ~0ull;

template <int NK, class L>
__device__ __forceinline__ void coop_lookup(const uint64_t* slots, const L& lay, const uint64_t (&off)[NK],
                                            const uint64_t (&tag)[NK], uint64_t* scratch, int lane,
                                            uint64_t (&out)[NK]) {
  constexpr int R = 4 * NK;
  static_assert(64 * NK <= kLookupScratch, "scratch holds one value per key");
  const int g = lane >> 2, sl = lane & 3;
  ulonglong2* ent = reinterpret_cast<ulonglong2*>(scratch);
  const char* base = reinterpret_cast<const char*>(slots) + 16 * sl;
  ulonglong2 sv[R];
  uint64_t tq[R];
#pragma unroll
  for (int i = 0; i < NK; i++) {
    ent[lane] = make_ulonglong2(off[i], tag[i]);
    wave_sync();
#pragma unroll
    for (int q = 4 * i; q < 4 * i + 4; q++) {
      const ulonglong2 e = ent[(q & 3) * 16 + g];
      tq[q] = e.y;
      sv[q] = *reinterpret_cast<const ulonglong2*>(base + e.x);
    }
    wave_sync();
  }
#pragma unroll
  for (int i = 0; i < NK; i++) scratch[64 * i + lane] = L::kNone;
  wave_sync();
#pragma unroll
  for (int q = 0; q < R; q++)
    if (sl == 3 && L::full(sv[q])) scratch[16 * q + g] = kLookupFull;
  wave_sync();
#pragma unroll
  for (int q = 0; q < R; q++) {
    uint64_t v;
    if (lay.match(sv[q], tq[q], v)) scratch[16 * q + g] = v;
  }
  wave_sync();
#pragma unroll
  for (int i = 0; i < NK; i++) out[i] = scratch[64 * i + lane];
  wave_sync();
}

// The count table's slots: the value is the raw count field.
struct CountLayout {
  static constexpr uint64_t kNone = 0;
  uint64_t kmo;
  uint32_t cshift;
  __device__ __forceinline__ bool match(const ulonglong2& s, uint64_t tag, uint64_t& v) const {
    const bool m0 = (s.x & kmo) == tag, m1 = (s.y & kmo) == tag;
    v = (m0 ? s.x : s.y) >> cshift;
    return m0 | m1;
  }
  static __device__ __forceinline__ bool full(const ulonglong2& s) { return s.y != 0; }
};

// Raw count field of a key whose home bucket is full and does not hold it (0 =
// absent): the buckets after it, each read whole, its slots compared without
// branches (about one absent key in twenty comes here at load 0.5).
__device__ __forceinline__ uint64_t table_field_after(const TableView& t, uint64_t tagged) {
  uint64_t b = bucket0(t, tagged & (t.occ - 1));
  for (uint32_t p = 1; p < t.max_probe; p++) {
    b = bucket_next(t, b);
    const ulonglong2* l2 = reinterpret_cast<const ulonglong2*>(t.slots + (b << 3));
    const ulonglong2 v[4] = {l2[0], l2[1], l2[2], l2[3]};
    uint64_t hit = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      hit = (v[j].x & t.kmo) == tagged ? v[j].x : hit;
      hit = (v[j].y & t.kmo) == tagged ? v[j].y : hit;
    }
    if (hit) return hit >> t.cshift;
    if (v[3].y == 0) return 0;
  }
  return 0;
}

// Counts of the keys (0 = absent or pruned; want[i] = false: 0).
template <int NK>
__device__ __forceinline__ void coop4_get(const TableView& t, const uint64_t (&key)[NK], const bool (&want)[NK],
                                          uint64_t* scratch, int lane, uint64_t (&out)[NK]) {
  uint64_t off[NK], tag[NK];
#pragma unroll
  for (int i = 0; i < NK; i++) {
    off[i] = want[i] ? bucket0(t, key[i]) << 6 : 0;
    tag[i] = want[i] ? key[i] | t.occ : 0;
  }
  coop_lookup<NK>(t.slots, CountLayout{t.kmo, t.cshift}, off, tag, scratch, lane, out);
#pragma unroll
  for (int i = 0; i < NK; i++) {
    out[i] = want[i] ? out[i] : 0;
    if (out[i] == kLookupFull) out[i] = table_field_after(t, tag[i]);
  }
  // all-ones fields: the count is in the side table
  bool side = false;
#pragma unroll
  for (int i = 0; i < NK; i++) side = side || out[i] == t.cmax;
  if (side) {
#pragma unroll
    for (int i = 0; i < NK; i++)
      if (out[i] == t.cmax) {
        const uint64_t* o = ovf_find(t, tag[i]);
        out[i] = o ? *o : out[i];
      }
  }
}

// Cooperative +1 of the 64 keys held one per lane (want = lane has a key).
// Eight lanes per key: in round q the lanes 8g..8g+7 read the eight slots of
// the home bucket of lane 8q+g's key (one coalesced 64-byte request per key,
// eight loads in flight per lane).  In each group the lane holding
// the key adds 1; otherwise the lowest empty slot of the snapshot is claimed
// with CAS.  The snapshot may be stale, but a slot's key never changes once
// set and every "empty" is confirmed by the CAS, so no key is inserted twice.
// All eight rounds' atomics are issued before any result is inspected, so a
// wavefront waits for one atomic round trip per 64 keys, not eight.
// Keys left unresolved (lost CAS race, full home bucket) are finished by
// their own lane with table_add; `spilled` reports a key that found no room
// within max_probe buckets.  Returns the number of new slots this lane
// claimed.
__device__ __forceinline__ uint32_t coop_add64(const TableView& t, uint64_t key, bool want,
                                               int lane, uint32_t* err, bool& spilled) {
  const uint64_t tagged = key | t.occ;
  const uint64_t b = bucket0(t, key);
  const int g = lane >> 3, sl = lane & 7;
  const uint64_t one = 1ull << t.cshift;
  uint64_t todo = __ballot(want);
  uint64_t sv[8], bq[8], tq[8], old[8];
#pragma unroll
  for (int q = 0; q < 8; q++) {
    bq[q] = __shfl(b, q * 8 + g);
    sv[q] = t.slots[(bq[q] << 3) + sl];
  }
  uint32_t kind = 0;  // per round, 2 bits: 1 = add issued, 2 = CAS issued
#pragma unroll
  for (int q = 0; q < 8; q++) {
    tq[q] = __shfl(tagged, q * 8 + g);
    old[q] = 0;
    const bool act = (todo >> (q * 8 + g)) & 1ull;
    const bool m = act && (sv[q] & t.kmo) == tq[q];
    const bool e = act && sv[q] == 0;
    const uint32_t mb = (uint32_t)((__ballot(m) >> (8 * g)) & 0xFFu);
    const uint32_t eb = (uint32_t)((__ballot(e) >> (8 * g)) & 0xFFu);
    unsigned long long* slot = (unsigned long long*)(t.slots + (bq[q] << 3) + sl);
    if (m) {
      old[q] = atomicAdd(slot, (unsigned long long)one);
      kind |= 1u << (2 * q);
    } else if (act && !mb && eb && sl == __builtin_ctz(eb)) {
      old[q] = atomicCAS(slot, 0ULL, (unsigned long long)(tq[q] | one));
      kind |= 2u << (2 * q);
    }
  }
  uint32_t claimed = 0;
  uint64_t carry = 0;  // bit w: the +1 of lane w's key wrapped its count field
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const uint32_t kq = (kind >> (2 * q)) & 3u;
    bool done = false, wrap = false;
    if (kq == 1u) {
      wrap = (old[q] >> t.cshift) == t.cmax;
      done = true;
    } else if (kq == 2u) {
      if (old[q] == 0) {
        claimed++;
        done = true;
      } else if ((old[q] & t.kmo) == tq[q]) {
        unsigned long long* slot = (unsigned long long*)(t.slots + (bq[q] << 3) + sl);
        const uint64_t o2 = atomicAdd(slot, (unsigned long long)one);
        wrap = (o2 >> t.cshift) == t.cmax;
        done = true;
      }
    }
    const uint32_t gd = byte_any8(__ballot(done));
    todo &= ~((uint64_t)gd << (8 * q));
    carry |= (uint64_t)byte_any8(__ballot(wrap)) << (8 * q);
  }
  // the key's own lane records a carry in its own table's side table
  if ((carry >> lane) & 1ull) ovf_add(t, tagged, t.cmax + 1, err);
  spilled = false;
  if ((todo >> lane) & 1ull) {
    const uint32_t r = table_add(t, key, 1, err);
    if (r == 2u) spilled = true;
    else claimed += r;
  }
  return claimed;
}

// Cooperative +1 of the 64 keys held one per lane, four lanes per key (the
// round layout of coop4_get: in round q the lanes 4g..4g+3 hold the sixteen
// bytes 16*sl.. of the home bucket of key 16q+g, lane 16q+g's key).  In each
// group the lane holding the key adds 1 to it; otherwise the lowest empty
// slot of the snapshot is claimed with CAS.  Same protocol and guarantees as
// coop_add64 (no key inserted twice; all rounds' atomics in flight before any
// result is inspected; unresolved keys finished by their own lane).
// `c` (1 <= c <= cmax) is the number of occurrences the lane adds.
__device__ __forceinline__ uint32_t coop4_add(const TableView& t, uint64_t key, bool want, int lane,
                                              uint32_t* err, bool& spilled, uint64_t c = 1) {
  const uint64_t tagged = key | t.occ;
  const uint64_t b = bucket0(t, key);
  const int g = lane >> 2, sl = lane & 3;
  const uint64_t one = c << t.cshift;
  uint64_t todo = __ballot(want);
  ulonglong2 sv[4];
  uint64_t bq[4], tq[4], old[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    bq[q] = __shfl(b, q * 16 + g);
    sv[q] = reinterpret_cast<const ulonglong2*>(t.slots + (bq[q] << 3))[sl];
  }
  uint32_t kind = 0;  // per round, 3 bits: 1 = add issued, 2 = CAS issued; bit 2 = second slot
#pragma unroll
  for (int q = 0; q < 4; q++) {
    tq[q] = __shfl(tagged, q * 16 + g);
    old[q] = 0;
    const bool act = (todo >> (q * 16 + g)) & 1ull;
    const bool m0 = act && (sv[q].x & t.kmo) == tq[q];
    const bool m1 = act && (sv[q].y & t.kmo) == tq[q];
    const bool e0 = act && sv[q].x == 0;
    const bool e1 = act && sv[q].y == 0;
    const uint32_t mb = (uint32_t)((__ballot(m0 | m1) >> (4 * g)) & 0xFu);
    const uint32_t eb = (uint32_t)((__ballot(e0 | e1) >> (4 * g)) & 0xFu);
    const uint64_t oneq = __shfl(one, q * 16 + g);
    if (m0 | m1) {
      const int j = m0 ? 0 : 1;
      old[q] = atomicAdd((unsigned long long*)(t.slots + (bq[q] << 3) + 2 * sl + j), (unsigned long long)oneq);
      kind |= (1u | ((uint32_t)j << 2)) << (3 * q);
    } else if (act && !mb && eb && sl == __builtin_ctz(eb)) {
      const int j = e0 ? 0 : 1;
      old[q] = atomicCAS((unsigned long long*)(t.slots + (bq[q] << 3) + 2 * sl + j), 0ULL,
                         (unsigned long long)(tq[q] | oneq));
      kind |= (2u | ((uint32_t)j << 2)) << (3 * q);
    }
  }
  uint32_t claimed = 0;
  uint64_t carry = 0;  // bit w: the +1 of lane w's key wrapped its count field
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const uint32_t kq = (kind >> (3 * q)) & 3u;
    const int j = (kind >> (3 * q + 2)) & 1u;
    bool done = false, wrap = false;
    const uint64_t cq = __shfl(c, q * 16 + g);
    if (kq == 1u) {
      wrap = (old[q] >> t.cshift) + cq > t.cmax;
      done = true;
    } else if (kq == 2u) {
      if (old[q] == 0) {
        claimed++;
        done = true;
      } else if ((old[q] & t.kmo) == tq[q]) {
        const uint64_t o2 = atomicAdd((unsigned long long*)(t.slots + (bq[q] << 3) + 2 * sl + j),
                                      (unsigned long long)(cq << t.cshift));
        wrap = (o2 >> t.cshift) + cq > t.cmax;
        done = true;
      }
    }
    todo &= ~((uint64_t)nibble_bits(__ballot(done)) << (16 * q));
    carry |= (uint64_t)nibble_bits(__ballot(wrap)) << (16 * q);
  }
  if ((carry >> lane) & 1ull) ovf_add(t, tagged, t.cmax + 1, err);
  spilled = false;
  if ((todo >> lane) & 1ull) {
    const uint32_t r = table_add(t, key, c, err);
    if (r == 2u) spilled = true;
    else claimed += r;
  }
  return claimed;
}

// Locality sort key of a read, fed its bases in order: bits 39..8 hold the
// smallest mixed hash over its canonical 16-mers (a minimizer; an N base
// reads as A, the key only orders reads), bits 7..0 the read's start relative
// to that 16-mer on the 16-mer's canonical strand.  Reads that share the
// minimizer overlap one locus of the transcriptome and sort by where they
// start along it, so neighbours in the order share most k-mers: their table
// lines are then reused from L2, and their windows merge before counting.
// Reads shorter than 16 bases sort last.
struct MinKey {
  uint32_t f = 0, r = 0, best = 0xFFFFFFFFu, bpos = 0;
  bool bfwd = true;
  __device__ __forceinline__ void push(uint32_t b, uint32_t pos) {
    f = (f << 2) | b;
    r = (r >> 2) | ((3u - b) << 30);
    if (pos >= 15) {
      const bool fw = f <= r;
      uint32_t x = fw ? f : r;
      x *= 0x9E3779B1u;
      x ^= x >> 16;
      x *= 0x85EBCA6Bu;
      x ^= x >> 13;
      if (x < best) {
        best = x;
        bpos = pos - 15;
        bfwd = fw;
      }
    }
  }
  __device__ __forceinline__ uint64_t key(uint32_t L) const {
    uint32_t rel = bfwd ? bpos : L - 16 - bpos;
    rel = rel > 255u ? 255u : rel;
    return ((uint64_t)best << 8) | (255u - rel);
  }
};
constexpr int kOrderKeyBits = 40;

}  // namespace tk
