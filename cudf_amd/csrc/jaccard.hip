// jaccard_index for gfx950.
//
// The reference (cpp/src/text/jaccard.cu) hashes the character windows of both columns into two
// chars-sized temporaries, sorts each row's hashes with a device-wide segmented sort, and counts unique
// and common values with a warp per row (66-170, 196-400).
//
// Here a row pair needs no sort and no temporary: the window hashes of both rows go into ONE open-addressing set in
// LDS with two membership bits per slot, "seen in row 1" and "seen in row 2".  |A|, |B| and |A n B| are then population
// counts of the two bit arrays and of their AND.
//
// What bounds it: LDS traffic and the vector instructions of hash and probe, about as much of each; HBM sees the chars
// once.  Hence
//   * buckets of four slots, read with one 16-byte LDS read: a hash that is there already (text repeats its words, and
//     the two rows are near-duplicates more often than not) costs that read and no compare-and-swap, and a probe seldom
//     goes on to a second bucket, for which the whole wavefront would wait;
//   * the membership bit is or-ed without asking for the old value: nothing waits for it;
//   * sets of five sizes, the smallest that holds a pair: what a CU can hide of the LDS latency is the number of
//     wavefronts that its 160 KB of sets allow.  A wavefront sizes the pairs, does the shortest itself, each with a set
//     of its own, and lists the others, each for the kernel with the set that fits it;
//   * a pair too long for one set in LDS is cut by hash value into up to kMaxParts parts of equal size, a workgroup each,
//     which hash the whole pair and keep their part (hashing is the cheap half); the counts of the parts add up.  Only
//     pairs beyond that use a set in global memory, whose atomics run at a fiftieth of the rate (1,600 such pairs among
//     250,000 of 2 KB rows: 3.7 of the call's 9.6 ms before the parts).
// 250,001 pairs of 2 KB rows (1.02 GB): 9.6 ms with a compare-and-swap on every window and four sizes of sets, 4.4 ms
// now (230 GB/s); about 100 vector instructions per 64 windows, a quarter of them the hash, issued in 70 % of the cycles.
#include "common.cuh"
#include "murmur.cuh"
#include "windows.cuh"

#include <algorithm>
#include <limits>

namespace nvtext_amd {
namespace {

// The tiers: slots of the set, wavefronts that share it, and the most bytes of a pair, which keep the load at or below
// 0.8 when no window repeats.
constexpr int kTiers              = 5;
constexpr uint32_t kSlots[kTiers] = {1024, 4096, 8064, 14336, 29440};
constexpr int kTierWaves[kTiers]  = {1, 4, 8, 8, 16};  // 7, 27, 53, 80 and 163 KB of LDS a workgroup
constexpr int64_t most_bytes(uint32_t slots) { return static_cast<int64_t>(slots) * 4 / 5; }
// the lists of pairs: tiers 1 to 4 (list = tier - 1), pairs in parts, pairs for the set in global memory
constexpr int kPartsList  = kTiers - 1;
constexpr int kGlobalList = kTiers;
constexpr int kLists      = kTiers + 1;

constexpr int64_t kPartBytes = 20000;  // bytes of a pair per part: 0.68 of the largest set, room for an uneven cut
constexpr int64_t kMaxParts  = 16;     // the hashing is done once per part

__device__ __host__ __forceinline__ int64_t parts_of(int64_t bytes) { return (bytes + kPartBytes - 1) / kPartBytes; }

__device__ __forceinline__ int list_of(int64_t bytes)
{
  int list = 0;
#pragma unroll
  for (int t = 1; t < kTiers; ++t) list += bytes > most_bytes(kSlots[t]);
  return list < kPartsList ? list : parts_of(bytes) <= kMaxParts ? kPartsList : kGlobalList;
}

// An insert-only set of non-zero uint32 values, in buckets of four slots that fill from the first to the last.  Beside it
// a bit array for each row: bit s says that the value in slot s occurs there.
// Where the set lies in global memory (IN_LDS false), reads of it go past the CU's own cache, which does not see what
// the atomics changed.
template <bool IN_LDS>
__device__ __forceinline__ uint32_t set_word(const uint32_t* p)
{
  if (IN_LDS) return *p;
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool IN_LDS>
struct PairSet {
  uint32_t* slots;   // 0 = empty; 16-byte aligned
  uint32_t buckets;

  __device__ __forceinline__ uint32_t home(uint32_t h) const { return __umulhi(h * 0x9E3779B1u, buckets); }

  // One look at one bucket for each of N values: `done` where the value is in the set now, and
  // its row's bit set; `taken` is 1 where the bucket is full of others, else 0.
  template <int N>
  __device__ __forceinline__ void insert_at(const bool (&want)[N], const uint32_t (&h)[N], const uint32_t (&bucket)[N], uint32_t* in, bool (&done)[N], uint32_t (&taken)[N]) const
  {
    uint32_t s[N], old[N];
    uint4 v[N];
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = read(bucket[k]);
#pragma unroll
    for (int k = 0; k < N; ++k) {
      // a_j: 1 as long as slots 0 .. j hold other values (min(v, v ^ h) is 0 where the slot is empty or holds h)
      uint32_t const a0 = min(min(1u, v[k].x), v[k].x ^ h[k]);
      uint32_t const a1 = min(min(a0, v[k].y), v[k].y ^ h[k]);
      uint32_t const a2 = min(min(a1, v[k].z), v[k].z ^ h[k]);
      uint32_t const a3 = min(min(a2, v[k].w), v[k].w ^ h[k]);
      s[k]     = 4u * bucket[k] + (a0 + a1 + a2);
      taken[k] = a3;
      done[k]  = want[k] && a3 == 0u;
    }
    // (also where the slot holds h already: cheaper than telling the two apart first)
#pragma unroll
    for (int k = 0; k < N; ++k)
      if (done[k]) old[k] = atomicCAS(&slots[s[k]], 0u, h[k]);
#pragma unroll
    for (int k = 0; k < N; ++k) {
      done[k] = done[k] && (old[k] == 0u || old[k] == h[k]);  // else another value came first
      if (done[k]) atomicOr(&in[s[k] >> 5], 1u << (s[k] & 31u));
    }
  }

  __device__ __forceinline__ uint4 read(uint32_t bucket) const
  {
    uint4 v;
    if (IN_LDS) {
      v = reinterpret_cast<const uint4*>(slots)[bucket];
    } else {
      v.x = set_word<false>(&slots[4u * bucket]);
      v.y = set_word<false>(&slots[4u * bucket + 1u]);
      v.z = set_word<false>(&slots[4u * bucket + 2u]);
      v.w = set_word<false>(&slots[4u * bucket + 3u]);
    }
    return v;
  }

  // From a bucket on, until the value is in the set.  false: every bucket is full (a set sized by the bytes of its pair
  // has room for every window; a part of one, whose share of the hashes is only near the average, may not).
  __device__ __forceinline__ bool insert(uint32_t h, uint32_t* in) const
  {
    uint32_t const v[1] = {h};
    bool const want[1]  = {true};
    uint32_t bucket[1]  = {home(h)};
    for (uint32_t probes = 0; probes < buckets;) {
      uint32_t taken[1];
      bool done[1];
      insert_at<1>(want, v, bucket, in, done, taken);
      if (done[0]) return true;
      if (taken[0] != 0u) {
        ++probes;
        if (++bucket[0] == buckets) bucket[0] = 0u;
      }  // (else another value came first: once more, at most until the bucket is full)
    }
    return false;
  }
};

// A share of the hashes by value, for pairs that are cut into parts (other bits than the set's own multiplication uses).
struct Part {
  uint32_t part, parts;
  __device__ __forceinline__ bool holds(uint32_t h) const
  {
    return parts == 1u || __umulhi((h ^ (h >> 15)) * 0x85EBCA6Bu, parts) == part;
  }
};

// A wavefront's own LDS for the tile it hashes.
struct TileLds {
  alignas(16) uint32_t bytes[kTileWords];
  uint16_t chars[kCharList];
  uint32_t later[kTile + kWave / 2];  // hashes that a first look at their bucket did not place
};

__device__ __forceinline__ float index_of(uint32_t count1, uint32_t count2, uint32_t intersects)
{
  int32_t const unions = static_cast<int32_t>(count1 + count2 - intersects);  // jaccard.cu:414-425
  return unions ? static_cast<float>(static_cast<int32_t>(intersects)) / static_cast<float>(unions) : 0.f;
}

// Where the rows of a pair are; null rows and empty rows have no hashes (jaccard.cu:211-220).
struct Pair {
  int64_t o1, n1, o2, n2;
  __device__ __forceinline__ int64_t bytes() const { return n1 + n2; }
};
__device__ __forceinline__ Pair pair_at(ColView const& c1, ColView const& c2, int64_t r)
{
  Pair p{0, 0, 0, 0};
  if (c1.valid(r)) {
    p.o1 = c1.off(r);
    p.n1 = c1.off(r + 1) - p.o1;
  }
  if (c2.valid(r)) {
    p.o2 = c2.off(r);
    p.n2 = c2.off(r + 1) - p.o2;
  }
  return p;
}

// The pair of a row number that is the same in every lane, through scalar loads (nothing that the kernels write is read
// here): what is computed from it and what branches on it is scalar as well.
__device__ __forceinline__ int64_t scalar_off(ColView const& c, int64_t i)
{
  using Long = const __attribute__((address_space(4))) int64_t*;
  using Int  = const __attribute__((address_space(4))) int32_t*;
  return c.is64 ? reinterpret_cast<Long>(reinterpret_cast<uintptr_t>(c.offsets))[i + c.offset]
                : static_cast<int64_t>(reinterpret_cast<Int>(reinterpret_cast<uintptr_t>(c.offsets))[i + c.offset]);
}
__device__ __forceinline__ bool scalar_valid(ColView const& c, int64_t i)
{
  if (!c.use_mask) return true;
  int64_t const b = i + c.offset;
  return (reinterpret_cast<const __attribute__((address_space(4))) uint32_t*>(reinterpret_cast<uintptr_t>(c.mask))[b >> 5] >> (b & 31)) & 1u;
}
__device__ __forceinline__ Pair uniform_pair_at(ColView const& c1, ColView const& c2, uint32_t row)
{
  int64_t const r = static_cast<int64_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(row))));
  Pair p{0, 0, 0, 0};
  if (scalar_valid(c1, r)) {
    p.o1 = scalar_off(c1, r);
    p.n1 = scalar_off(c1, r + 1) - p.o1;
  }
  if (scalar_valid(c2, r)) {
    p.o2 = scalar_off(c2, r);
    p.n2 = scalar_off(c2, r + 1) - p.o2;
  }
  return p;
}

// Slots for a pair: room for twice its windows, which are at most its bytes, or what the tier has (whole words of bits).
__device__ __forceinline__ uint32_t slots_for(int64_t bytes, uint32_t most)
{
  return static_cast<uint32_t>(min(static_cast<int64_t>(most), (2 * bytes + 63) / 32 * 32));
}

// ... and in global memory: room for one and a half times its windows.
__device__ __host__ __forceinline__ uint64_t slots_for_global(int64_t bytes)
{
  uint64_t s = 64;
  while (2 * s < 3 * static_cast<uint64_t>(bytes)) s <<= 1;
  return s;
}

// Hashes the windows of both rows (jaccard.cu:249-292) and inserts the non-zero hashes into the set.  The tiles of the
// two rows, one list, go to `nwaves` wavefronts in turn; those of a short pair are cut finer than kTile so that each has
// one.  false: the set was full.
// Nearly every hash finds its place with one look at one bucket, but in most rounds of 64 some lane does not: those are
// put aside and placed 64 at a time, so that a round does not wait for its slowest lane.
template <bool IN_LDS>
__device__ __forceinline__ bool insert_pair(ColView const& c1, ColView const& c2, Pair const& pair, int32_t width, PairSet<IN_LDS> const& set,
                                            uint32_t* in1, uint32_t* in2, Part part, TileLds& lds, int wave, int nwaves, int lane)
{
  auto const hash = [](auto const& src, uint32_t len, auto& h) { murmur3_x86_32_unmixed(src, len, 0u, h); };  // jaccard.cu:258: seed 0
  bool ok         = true;
  if (static_cast<int64_t>(width) * 4 <= kHalo) {
    int64_t const even   = pair.bytes() / (nwaves * kWave) * kWave;
    int32_t const tile   = static_cast<int32_t>(min(max(even, static_cast<int64_t>(kWave)), static_cast<int64_t>(kTile)));
    int64_t const tiles1 = (pair.n1 + tile - 1) / tile, tiles = tiles1 + (pair.n2 + tile - 1) / tile;
    uint32_t later = 0, later1 = 0;  // hashes put aside, and how many of them (the first ones) are row 1's: the same in every lane
    for (int64_t t = wave; t < tiles; t += nwaves) {
      bool const second      = t >= tiles1;
      const uint8_t* const r = second ? c2.chars + pair.o2 : c1.chars + pair.o1;
      int64_t const n        = second ? pair.n2 : pair.n1;
      uint32_t* const in     = second ? in2 : in1;
      int64_t const base     = (second ? t - tiles1 : t) * tile;
      uint32_t const cnt     = static_cast<uint32_t>(min(static_cast<int64_t>(tile), n - base));
      hash_tile_windows<uint32_t>(r, n, base, cnt, width, lds.bytes, lds.chars, lane, hash, [&](auto const& valid, auto const& hv) {
        constexpr int N = sizeof(hv) / sizeof(hv[0]);
        bool want[N], done[N];
        uint32_t bucket[N], taken[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
          want[k]   = valid[k] && hv[k] != 0u && part.holds(hv[k]);  // 282-286: zero hashes are dropped
          bucket[k] = set.home(hv[k]);
        }
        set.template insert_at<N>(want, hv, bucket, in, done, taken);
#pragma unroll
        for (int k = 0; k < N; ++k) {
          bool const left      = want[k] && !done[k];
          uint64_t const which = ballot64(left);
          if (left) lds.later[later + lanes_below(which)] = hv[k];
          later += static_cast<uint32_t>(__builtin_popcountll(which));
        }
      });
      if (!second) later1 = later;
      if (later >= kWave / 2 || t + nwaves >= tiles) {
        for (uint32_t i = lane; i < later; i += kWave) ok = set.insert(lds.later[i], i < later1 ? in1 : in2) && ok;
        later = later1 = 0;
      }
    }
    return ok;
  }
  // very wide windows: bytes straight from global memory
#pragma nounroll
  for (int row = 0; row < 2; ++row) {
    const uint8_t* const r = row == 0 ? c1.chars + pair.o1 : c2.chars + pair.o2;
    int64_t const n        = row == 0 ? pair.n1 : pair.n2;
    for (int64_t gpos = static_cast<int64_t>(wave) * kWave + lane; gpos < n; gpos += nwaves * kWave) {
      int64_t const remaining = n - gpos;
      BoundedSrc const src[1] = {{r + gpos, remaining}};
      uint32_t hlen;
      uint32_t const readable = static_cast<uint32_t>(min(remaining, static_cast<int64_t>(width) * 4));
      if (window_at(src[0], r + gpos, remaining, readable, gpos == 0, false, width, &hlen)) {
        uint32_t hv[1];
        hash(src, hlen, hv);
        if (hv[0] != 0u && part.holds(hv[0])) ok = set.insert(hv[0], row == 0 ? in1 : in2) && ok;
      }
    }
  }
  return ok;
}

template <int WAVES>
struct PairScratch {
  TileLds tile[WAVES];
  uint32_t sums[3][WAVES];
  uint32_t full;
};

// One row pair (or a part of it) by WAVES wavefronts with a set of `nslots` slots (a multiple of 32): clears
// the set, inserts both rows, counts.  The counts are thread 0's; false (everywhere) when the set was full.
template <int WAVES, bool IN_LDS>
__device__ __forceinline__ bool count_pair(ColView const& c1, ColView const& c2, Pair const& pair, int32_t width, Part part, uint32_t* slots,
                                           uint32_t* in1, uint32_t* in2, uint32_t nslots, PairScratch<WAVES>& scratch, uint32_t (&counts)[3])
{
  constexpr uint32_t kPairThreads = WAVES * kWave;
  int const lane = lane_id();
  int const wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
  // (the arrays are 16-byte aligned: whole uint4 stores)
  for (uint32_t i = threadIdx.x; i < nslots / 4; i += kPairThreads) reinterpret_cast<uint4*>(slots)[i] = make_uint4(0u, 0u, 0u, 0u);
  for (uint32_t i = threadIdx.x; i < nslots / 32; i += kPairThreads) {
    in1[i] = 0u;
    in2[i] = 0u;
  }
  if (threadIdx.x == 0) scratch.full = 0u;
  __syncthreads();
  PairSet<IN_LDS> const set{slots, nslots / 4};
  bool const ok = insert_pair(c1, c2, pair, width, set, in1, in2, part, scratch.tile[wave], wave, WAVES, lane);
  if (!ok) scratch.full = 1u;
  __syncthreads();
  uint32_t u[3] = {0, 0, 0};
  for (uint32_t i = threadIdx.x; i < nslots / 32; i += kPairThreads) {
    uint32_t const a = set_word<IN_LDS>(&in1[i]), b = set_word<IN_LDS>(&in2[i]);
    u[0] += __builtin_popcount(a);
    u[1] += __builtin_popcount(b);
    u[2] += __builtin_popcount(a & b);
  }
  if (IN_LDS) {  // (a wavefront's counts fit 16 bits: two sums in one)
    u[0] = wave_inclusive_scan(u[0] | (u[1] << 16));
    u[1] = u[0] >> 16;
    u[0] &= 0xFFFFu;
    u[2] = wave_inclusive_scan(u[2]);
  } else {
    for (int k = 0; k < 3; ++k) u[k] = wave_inclusive_scan(u[k]);
  }
  if (lane == kWave - 1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) scratch.sums[k][wave] = u[k];
  }
  bool const full = scratch.full != 0u;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    counts[k] = 0;
    for (int w = 0; w < WAVES; ++w) counts[k] += scratch.sums[k][w];
  }
  // (the next pair's set is cleared by now at most: what it overwrites of `scratch` it overwrites after its own barrier)
  return !full;
}

// Work lists in `work`: a header of 16 words -- [i] = pairs on list i, [kLists] = null rows of the result,
// [8..9] = the most bytes a pair of the global list has (64 bits) -- then four counters (|A|, |B|, |A n B|, parts done) for
// every entry of the list of pairs in parts, and `rows` entries for each list.
constexpr int kListHeader = 16;
constexpr int32_t kLookRows = 32768;  // see nvtext_amd_jaccard_index
__host__ __device__ __forceinline__ size_t work_words(int64_t rows) { return kListHeader + static_cast<size_t>(kLists + 4) * static_cast<size_t>(rows); }
__device__ __forceinline__ uint32_t* list_entries(uint32_t* work, int list, int64_t rows) { return work + kListHeader + (4 + list) * rows; }
__device__ __forceinline__ uint32_t* part_counters(uint32_t* work) { return work + kListHeader; }
__device__ __forceinline__ void list_for_global(uint32_t* work, int64_t rows, int64_t r, int64_t bytes)
{
  list_entries(work, kGlobalList, rows)[atomicAdd(&work[kGlobalList], 1u)] = static_cast<uint32_t>(r);
  atomicMax(reinterpret_cast<unsigned long long*>(&work[8]), static_cast<unsigned long long>(bytes));
}

struct WaveSetLds {
  alignas(16) uint32_t slots[kSlots[0]];
  uint32_t in1[kSlots[0] / 32], in2[kSlots[0] / 32];
  TileLds tile;
};

// A workgroup sizes `per_group` consecutive pairs at once (at most kThreads: threads <-> pairs, coalesced offset loads),
// lists those that need more than a wavefront's own set for the later kernels with one atomic per list (atomics on one
// cache line run at about 150 M/s: one per wavefront and list was most of this kernel's time), and its wavefronts do the
// others, each taking the next one when it is done with one.  A column of few pairs is shared out over more workgroups.
__global__ void __launch_bounds__(kThreads) jaccard_wave_kernel(ColView c1, ColView c2, int32_t width, float* __restrict__ out,
                                                                uint32_t* __restrict__ work, int per_group)
{
  __shared__ WaveSetLds lds_all[kWaves];
  __shared__ uint32_t listed[kLists], place[kLists], solo[kThreads], solos, next;
  int const lane     = lane_id();
  int const wave     = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
  WaveSetLds& lds    = lds_all[wave];
  int64_t const rows = c1.size;
  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  for (int64_t base = static_cast<int64_t>(blockIdx.x) * per_group; base < rows; base += static_cast<int64_t>(gridDim.x) * per_group) {
    __syncthreads();
    if (threadIdx.x < kLists) listed[threadIdx.x] = 0u;
    if (threadIdx.x == 0) solos = next = 0u;
    __syncthreads();
    int64_t const r   = base + threadIdx.x;
    bool const have   = r < rows && static_cast<int>(threadIdx.x) < per_group;
    int64_t const all = have ? pair_at(c1, c2, r).bytes() : 0;
    bool const later  = have && all > most_bytes(kSlots[0]);
    int const list    = list_of(all);
    uint32_t at       = 0;
    if (have && !later) solo[atomicAdd(&solos, 1u)] = static_cast<uint32_t>(r);
    if (later) at = atomicAdd(&listed[list], 1u);
    __syncthreads();
    if (threadIdx.x < kLists && listed[threadIdx.x] != 0u) place[threadIdx.x] = atomicAdd(&work[threadIdx.x], listed[threadIdx.x]);
    __syncthreads();
    if (later) {
      at += place[list];
      list_entries(work, list, rows)[at] = static_cast<uint32_t>(r);
      if (list == kPartsList) reinterpret_cast<uint4*>(part_counters(work))[at] = make_uint4(0u, 0u, 0u, 0u);
      if (list == kGlobalList) atomicMax(reinterpret_cast<unsigned long long*>(&work[8]), static_cast<unsigned long long>(all));
    }
    for (;;) {
      uint32_t t = 0;
      if (lane == 0) t = atomicAdd(&next, 1u);
      t = wave_bcast(t, 0);
      if (t >= solos) break;
      uint32_t const pr     = solo[t];
      Pair const q          = uniform_pair_at(c1, c2, pr);
      uint32_t const nslots = slots_for(q.bytes(), kSlots[0]);
      for (uint32_t i = lane; i < nslots / 4; i += kWave) reinterpret_cast<uint4*>(lds.slots)[i] = make_uint4(0u, 0u, 0u, 0u);
      if (static_cast<uint32_t>(lane) < nslots / 32) {
        lds.in1[lane] = 0u;
        lds.in2[lane] = 0u;
      }
      wave_sync();
      PairSet<true> const set{lds.slots, nslots / 4};
      insert_pair(c1, c2, q, width, set, lds.in1, lds.in2, Part{0, 1}, lds.tile, 0, 1, lane);  // (the set has room for every window)
      wave_sync();
      uint32_t u1 = 0, both = 0;
      if (static_cast<uint32_t>(lane) < nslots / 32) {  // at most 32 words of bits
        uint32_t const a = lds.in1[lane], b = lds.in2[lane];
        u1   = __builtin_popcount(a) | (static_cast<uint32_t>(__builtin_popcount(b)) << 16);
        both = __builtin_popcount(a & b);
      }
      u1   = wave_inclusive_scan(u1);  // (at most 1024 in either half)
      both = wave_inclusive_scan(both);
      if (lane == kWave - 1) out[pr] = index_of(u1 & 0xFFFFu, u1 >> 16, both);
      wave_sync();
    }
  }
}

// The pairs of a tier's list, one workgroup of WAVES wavefronts and one set of SLOTS slots per pair.
template <int TIER>
__global__ void __launch_bounds__(kTierWaves[TIER] * kWave) jaccard_listed_kernel(ColView c1, ColView c2, int32_t width, float* __restrict__ out,
                                                                                  uint32_t* __restrict__ work)
{
  constexpr uint32_t SLOTS = kSlots[TIER];
  constexpr int WAVES      = kTierWaves[TIER];
  __shared__ alignas(16) uint32_t slots[SLOTS];
  __shared__ uint32_t in1[SLOTS / 32], in2[SLOTS / 32];
  __shared__ PairScratch<WAVES> scratch;
  int64_t const rows   = c1.size;
  uint32_t const count = work[TIER - 1];
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    uint32_t const r      = list_entries(work, TIER - 1, rows)[i];
    Pair const pair       = uniform_pair_at(c1, c2, r);
    uint32_t const nslots = slots_for(pair.bytes(), SLOTS);
    uint32_t counts[3];
    count_pair<WAVES, true>(c1, c2, pair, width, Part{0, 1}, slots, in1, in2, nslots, scratch, counts);
    if (threadIdx.x == 0) out[r] = index_of(counts[0], counts[1], counts[2]);
  }
}

// The pairs in parts: workgroup (x, y) does part y of the pairs x, x + gridDim.x, ...  The last part to be done writes
// the index.  A part whose set is full (its share of the hashes far above the average) has the pair done once more, by
// the set in global memory.
constexpr int kPartsTier = kTiers - 1;
__global__ void __launch_bounds__(kTierWaves[kPartsTier] * kWave) jaccard_parts_kernel(ColView c1, ColView c2, int32_t width, float* __restrict__ out,
                                                                                       uint32_t* __restrict__ work)
{
  constexpr uint32_t SLOTS = kSlots[kPartsTier];
  constexpr int WAVES      = kTierWaves[kPartsTier];
  __shared__ alignas(16) uint32_t slots[SLOTS];
  __shared__ uint32_t in1[SLOTS / 32], in2[SLOTS / 32];
  __shared__ PairScratch<WAVES> scratch;
  int64_t const rows   = c1.size;
  uint32_t const count = work[kPartsList];
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    uint32_t const r  = list_entries(work, kPartsList, rows)[i];
    Pair const pair   = uniform_pair_at(c1, c2, r);
    Part const part{blockIdx.y, static_cast<uint32_t>(parts_of(pair.bytes()))};
    if (part.part >= part.parts) continue;
    uint32_t counts[3];
    bool const ok = count_pair<WAVES, true>(c1, c2, pair, width, part, slots, in1, in2, SLOTS, scratch, counts);
    if (threadIdx.x == 0) {
      uint32_t* const at = part_counters(work) + 4 * static_cast<int64_t>(i);
      for (int k = 0; k < 3; ++k) atomicAdd(&at[k], counts[k]);
      __threadfence();
      // a full set leaves a mark far above the number of parts
      uint32_t const done = atomicAdd(&at[3], ok ? 1u : 1u + (1u << 16)) + (ok ? 1u : 1u + (1u << 16));
      if ((done & 0xFFFFu) == part.parts) {
        __threadfence();
        if (done >> 16)
          list_for_global(work, rows, r, pair.bytes());
        else
          out[r] = index_of(atomicAdd(&at[0], 0u), atomicAdd(&at[1], 0u), atomicAdd(&at[2], 0u));
      }
    }
  }
}

// The listed pairs, each workgroup with its own set in global memory (`table_slots` slots, then the two bit arrays).
__global__ void __launch_bounds__(kThreads) jaccard_global_kernel(ColView c1, ColView c2, int32_t width, float* __restrict__ out,
                                                                  uint32_t* __restrict__ work, uint32_t* __restrict__ tables,
                                                                  uint64_t table_slots)
{
  __shared__ PairScratch<kWaves> scratch;
  int64_t const rows   = c1.size;
  uint32_t const count = work[kGlobalList];
  uint32_t* const mine = tables + static_cast<uint64_t>(blockIdx.x) * (table_slots + 2 * (table_slots / 32));
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    uint32_t const r    = list_entries(work, kGlobalList, rows)[i];
    Pair const pair     = uniform_pair_at(c1, c2, r);
    uint32_t const need = static_cast<uint32_t>(slots_for_global(pair.bytes()));
    uint32_t counts[3];
    count_pair<kWaves, false>(c1, c2, pair, width, Part{0, 1}, mine, mine + table_slots, mine + table_slots + table_slots / 32, need, scratch, counts);
    if (threadIdx.x == 0) out[r] = index_of(counts[0], counts[1], counts[2]);
    __syncthreads();
  }
}

// out[w] = validity word w of column 1 AND of column 2 (bits past `bits` are 0); *nulls += zero bits.
__global__ void and_bitmask_kernel(uint32_t* __restrict__ out, const uint32_t* __restrict__ m1, int32_t begin1, const uint32_t* __restrict__ m2,
                                   int32_t begin2, int32_t bits, int32_t words, uint32_t* __restrict__ nulls)
{
  int32_t const w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= words) return;
  auto word_of = [&](const uint32_t* m, int32_t begin) -> uint32_t {
    if (!m) return 0xFFFFFFFFu;
    int64_t const first = static_cast<int64_t>(begin) + static_cast<int64_t>(w) * 32;
    int64_t const sw    = first >> 5;
    int const sh        = static_cast<int>(first & 31);
    int64_t const last  = (static_cast<int64_t>(begin) + bits - 1) >> 5;
    uint32_t v          = m[sw] >> sh;
    if (sh != 0 && sw + 1 <= last) v |= m[sw + 1] << (32 - sh);
    return v;
  };
  uint32_t v              = word_of(m1, begin1) & word_of(m2, begin2);
  int32_t const remaining = bits - w * 32;
  uint32_t const live     = remaining < 32 ? (1u << remaining) - 1u : 0xFFFFFFFFu;
  v &= live;
  out[w] = v;
  uint32_t const zeros = __builtin_popcount(~v & live);
  if (zeros) atomicAdd(nulls, zeros);
}

__global__ void publish_header_kernel(const uint32_t* __restrict__ work, uint32_t* __restrict__ host, HostPost post)
{
  host[threadIdx.x] = work[threadIdx.x];
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) post.send();
}

}  // namespace
}  // namespace nvtext_amd

extern "C" {

nvtext_amd_status nvtext_amd_jaccard_index(const nvtext_amd_strings_column* input1, const nvtext_amd_strings_column* input2, int32_t width,
                                           void* stream_, const nvtext_amd_allocator* mr_, nvtext_amd_fixed_column* out)
{
  using namespace nvtext_amd;
  EntryScope const entry("nvtext_amd_jaccard_index");
  if (!input1 || !input2 || !out) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null argument");
  *out = nvtext_amd_fixed_column{};
  // cpp/src/text/jaccard.cu:441-446, same order and messages
  if (input1->size != input2->size) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "input columns must be the same size");
  if (width < 2) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "Parameter width should be an integer value of 2 or greater");
  for (const nvtext_amd_strings_column* c : {input1, input2}) {
    if (c->size < 0 || c->null_count < 0 || c->null_count > c->size) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "invalid column sizes");
    if (c->null_count > 0 && !c->null_mask) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null_count > 0 requires a null mask");
  }
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  Mr mr{mr_, stream};
  int32_t const rows = input1->size;
  out->type          = NVTEXT_AMD_TYPE_FLOAT32;
  out->size          = rows;
  if (rows == 0) return NVTEXT_AMD_SUCCESS;  // jaccard.cu:449: an empty FLOAT32 column

  out->data_bytes = static_cast<size_t>(rows) * sizeof(float);
  out->data       = mr.allocate(out->data_bytes);
  if (!out->data) return fail(NVTEXT_AMD_ALLOC_FAILED, "result allocation failed");
  bool const with_mask = input1->null_count > 0 || input2->null_count > 0;  // 471-476
  if (with_mask) {
    out->null_mask_bytes = mask_alloc_bytes(rows);
    out->null_mask       = static_cast<uint32_t*>(mr.allocate(out->null_mask_bytes));
    if (!out->null_mask) {
      nvtext_amd_fixed_column_free(out, stream_, mr_);
      return fail(NVTEXT_AMD_ALLOC_FAILED, "mask allocation failed");
    }
  }
  Temp work(mr, work_words(rows) * sizeof(uint32_t));
  if (!work.ok()) {
    nvtext_amd_fixed_column_free(out, stream_, mr_);
    return fail(NVTEXT_AMD_ALLOC_FAILED, "temporary allocation failed");
  }
  uint32_t* const lists = work.as<uint32_t>();
  launch_fill_u32(lists, 0u, kListHeader, stream);

  ColView const v1 = make_view(*input1);
  ColView const v2 = make_view(*input2);
  float* const values = static_cast<float*>(out->data);
  int const cus       = device_cus();
  {
    ProfileScope ps("jaccard_wave_kernel", stream);
    int per_group = kThreads;
    while (per_group > kWaves && rows / per_group < 4 * cus) per_group /= 2;
    int64_t const groups = (static_cast<int64_t>(rows) + per_group - 1) / per_group;
    unsigned const grid  = static_cast<unsigned>(std::min<int64_t>(groups, static_cast<int64_t>(cus) * 64));
    hipLaunchKernelGGL(jaccard_wave_kernel, dim3(grid), dim3(kThreads), 0, stream, v1, v2, width, values, lists, per_group);
  }
  if (with_mask) {
    int32_t const words = (rows + 31) / 32;
    hipLaunchKernelGGL(and_bitmask_kernel, dim3((words + 255) / 256), dim3(256), 0, stream, out->null_mask,
                       input1->null_count > 0 ? input1->null_mask : nullptr, input1->offset,
                       input2->null_count > 0 ? input2->null_mask : nullptr, input2->offset, rows, words, &lists[kLists]);
  }
  // what the host has to know: the header of the lists
  uint32_t copied[kListHeader] = {};
  uint64_t* const pinned       = host_scalars();
  const uint32_t* const head   = pinned ? reinterpret_cast<const uint32_t*>(pinned) : copied;
  auto const read_header       = [&]() -> hipError_t {
    if (!pinned) {
      hipError_t const e = hipMemcpyAsync(copied, lists, sizeof(copied), hipMemcpyDeviceToHost, stream);
      return e == hipSuccess ? hipStreamSynchronize(stream) : e;
    }
    HostPost const post = new_post();
    hipLaunchKernelGGL(publish_header_kernel, dim3(1), dim3(kListHeader), 0, stream, lists, reinterpret_cast<uint32_t*>(pinned), post);
    hipError_t const e = hipGetLastError();
    return e == hipSuccess ? wait_for_post(post, stream) : e;
  };
  // In a column of few pairs the launches of the other kernels, most of which would find their lists empty, are more than
  // the work: the host looks at the lists first and launches what has something to do (7 pairs of 300 bytes 48 -> 20 us).
  // In a larger one the wait costs more than a few empty launches.
  bool const look   = rows <= kLookRows;
  hipError_t e      = look ? read_header() : hipSuccess;
  auto const listed = [&](int list) { return look ? static_cast<int32_t>(head[list]) : rows; };
  auto const grid_of = [&](int list, int per_cu) { return dim3(static_cast<unsigned>(std::min<int64_t>(listed(list), static_cast<int64_t>(cus) * per_cu))); };
  if (e == hipSuccess && listed(0) > 0) {
    ProfileScope ps("jaccard_listed_kernel<1>", stream);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(jaccard_listed_kernel<1>), grid_of(0, 28), dim3(kTierWaves[1] * kWave), 0, stream, v1, v2, width, values, lists);
  }
  if (e == hipSuccess && listed(1) > 0) {
    ProfileScope ps("jaccard_listed_kernel<2>", stream);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(jaccard_listed_kernel<2>), grid_of(1, 12), dim3(kTierWaves[2] * kWave), 0, stream, v1, v2, width, values, lists);
  }
  if (e == hipSuccess && listed(2) > 0) {
    ProfileScope ps("jaccard_listed_kernel<3>", stream);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(jaccard_listed_kernel<3>), grid_of(2, 8), dim3(kTierWaves[3] * kWave), 0, stream, v1, v2, width, values, lists);
  }
  if (e == hipSuccess && listed(3) > 0) {
    ProfileScope ps("jaccard_listed_kernel<4>", stream);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(jaccard_listed_kernel<4>), grid_of(3, 4), dim3(kTierWaves[4] * kWave), 0, stream, v1, v2, width, values, lists);
  }
  bool const in_parts = listed(kPartsList) > 0;
  if (e == hipSuccess && in_parts) {
    ProfileScope ps("jaccard_parts_kernel", stream);
    hipLaunchKernelGGL(jaccard_parts_kernel, dim3(grid_of(kPartsList, 1).x, static_cast<unsigned>(kMaxParts)), dim3(kTierWaves[kPartsTier] * kWave), 0, stream,
                       v1, v2, width, values, lists);
  }
  if (e == hipSuccess && in_parts) e = read_header();  // (a part can turn out too full: its pair is then on the list of the last kernel)
  if (e != hipSuccess) {
    nvtext_amd_fixed_column_free(out, stream_, mr_);
    return fail(NVTEXT_AMD_DEVICE_ERROR, hipGetErrorString(e));
  }
  out->null_count = static_cast<int32_t>(head[kLists]);
  if (head[kGlobalList] > 0) {
    uint64_t const most  = (static_cast<uint64_t>(head[9]) << 32) | head[8];
    uint64_t const slots = slots_for_global(static_cast<int64_t>(most));
    if (slots > (uint64_t{1} << 31)) {
      nvtext_amd_fixed_column_free(out, stream_, mr_);
      return fail(NVTEXT_AMD_OVERFLOW, "a row pair is too long");
    }
    unsigned const grid = static_cast<unsigned>(std::min<uint64_t>(head[kGlobalList], static_cast<uint64_t>(cus)));
    Temp tables(mr, static_cast<size_t>(grid) * (slots + 2 * (slots / 32)) * sizeof(uint32_t));
    if (!tables.ok()) {
      nvtext_amd_fixed_column_free(out, stream_, mr_);
      return fail(NVTEXT_AMD_ALLOC_FAILED, "temporary allocation failed");
    }
    ProfileScope ps("jaccard_global_kernel", stream);
    hipLaunchKernelGGL(jaccard_global_kernel, dim3(grid), dim3(kThreads), 0, stream, v1, v2, width, values, lists, tables.as<uint32_t>(), slots);
    NVTEXT_HIP_TRY_OR(hipGetLastError(), nvtext_amd_fixed_column_free(out, stream_, mr_));
    // the tables are released in stream order when `tables` goes out of scope
  }
  NVTEXT_HIP_TRY_OR(hipGetLastError(), nvtext_amd_fixed_column_free(out, stream_, mr_));
  return NVTEXT_AMD_SUCCESS;
}

void nvtext_amd_fixed_column_free(nvtext_amd_fixed_column* col, void* stream, const nvtext_amd_allocator* mr)
{
  if (!col) return;
  nvtext_amd::Mr m{mr, static_cast<hipStream_t>(stream)};
  m.deallocate(col->data, col->data_bytes);
  m.deallocate(col->null_mask, col->null_mask_bytes);
  *col = nvtext_amd_fixed_column{};
}

}  // extern "C"
