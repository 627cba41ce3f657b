// jaccard_index for gfx950.
//
// The reference (cpp/src/text/jaccard.cu) hashes the character windows of both columns into two
// chars-sized temporaries, sorts each row's hashes with a device-wide segmented sort, and counts unique
// and common values with a warp per row (66-170, 196-400).
//
// Here a row pair needs no sort and no temporary: the window hashes of both rows go into ONE open-addressing set in
// LDS whose slots also say "seen in row 1" and "seen in row 2".  |A|, |B| and |A n B| are then counts of these marks.
//
// What bounds it: vector and scalar instructions, 70 and 62 per 64 windows, and LDS, each busy for 50 to 60 % of the time; HBM sees the
// chars once.  Hence
//   * buckets of four slots, read with one 16-byte LDS read: a probe seldom goes on to a second bucket, for which the whole
//     wavefront would wait; what one look does not place is put aside and placed 64 at a time;
//   * value and marks in one word (PackedSet): no address and no mask to be made for a mark;
//   * every wavefront of a pair hashes as many windows as the others, to 64, and the sets are left empty by the pass that
//     counts: two barriers a pair;
//   * sets of five sizes, the smallest that holds a pair: what a CU can hide of the LDS latency is the number of
//     wavefronts that its 160 KB of sets allow (as does the number of scalar registers: eight per SIMD have 96 each).  A
//     wavefront sizes the pairs, does the shortest itself, each with a set of its own, and lists the others, each for the
//     kernel with the set that fits it;
//   * a pair too long for one set in LDS is cut by hash value into up to kMaxParts parts of equal size, a workgroup each,
//     which hash the whole pair and keep their part (hashing is the cheap half); the counts of the parts add up.  Only
//     pairs beyond that use a set in global memory, whose atomics run at a fiftieth of the rate (1,600 such pairs among
//     250,000 of 2 KB rows: 3.7 of the call's 9.6 ms before the parts).
// 250,001 pairs of 2 KB rows (1.02 GB): 4.08 ms with whole values, bits in arrays and tiles in turn, 3.5 with a hundred vector instructions
// per 64 windows, 2.95 ms now (347 GB/s).
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
constexpr uint32_t kSlots[kTiers] = {1024, 4096, 7008, 15488, 29440};
constexpr int kTierWaves[kTiers]  = {1, 4, 8, 12, 16};  // 6, 23, 41, 81 and 144 KB of LDS a workgroup
constexpr int kSimdWaves[kTiers]  = {6, 7, 8, 6, 4};    // wavefronts per SIMD that these leave room for
static_assert(kSlots[kTiers - 1] / 4 <= 255 * kTierWaves[kTiers - 1] * kWave, "the counters of a lane");
constexpr int64_t most_bytes(uint32_t slots) { return static_cast<int64_t>(slots) * 4 / 5; }
// the lists of pairs: tiers 1 to 4 (list = tier - 1), pairs in parts, pairs for the set in global memory
constexpr int kPartsList  = kTiers - 1;
constexpr int kGlobalList = kTiers;
constexpr int kLists      = kTiers + 1;

constexpr int64_t kPartBytes = 20000;  // bytes of a pair per part: 0.68 of the largest set, room for an uneven cut
// The hashing is done once per part, and the parts of a pair on as many CUs: a pair of 330 KB in 17 parts 0.22 ms, with one set in
// global memory 3.7, and of 600 KB in 30 0.38 and 6.6; a thousand of them 13 and 42 ms, and 26 and 48 (with 64 parts many pairs
// of more than 640 KB would take longer).
constexpr int64_t kMaxParts  = 32;

__device__ __host__ __forceinline__ int64_t parts_of(int64_t bytes) { return (bytes + kPartBytes - 1) / kPartBytes; }

__device__ __forceinline__ int list_of(int64_t bytes)
{
  int list = 0;
#pragma unroll
  for (int t = 1; t < kTiers; ++t) list += bytes > most_bytes(kSlots[t]);
  return list < kPartsList ? list : parts_of(bytes) <= kMaxParts ? kPartsList : kGlobalList;
}

// Insert-only sets of non-zero uint32 values (products of hashes, see value_of), in buckets of four slots that fill from the first to
// the last.  A value's home bucket is what its top says.  place_at() has one look at bucket home + distance for each of
// N values: `left` stays where the value is not in the set now, marked as its row's; `taken` tells whether the bucket is full
// of others, so that the next one is to be looked at.
//
// The set of a pair whose windows LDS has room for.  A slot holds the low 24 bits of the value, which tell the values of one
// home bucket apart where there are 256 buckets and more, how many steps from home it lies (6 bits), and two bits that say
// which rows it occurs in: one compare-and-swap places a value and marks it, where that finds the value there already it is marked with
// an or of a constant to the same address, and counting is a pass over the slots.  (With whole values and the bits in arrays
// of their own a look took 65 vector instructions for 128 windows; now 50, beside 30 for the hashes of windows of five bytes.)
struct PackedSet {
  static constexpr uint32_t kValue    = 0x00FFFFFFu;
  static constexpr uint32_t kFar      = 64;  // steps from home that can be told
  static constexpr int kDistanceAt    = 25;
  static constexpr uint32_t kSame     = 0x7EFFFFFFu;  // value and distance
  static constexpr uint32_t kLeast    = 1024;         // slots
  using Mark                          = uint32_t;
  uint32_t* slots;  // 0 = empty; 16-byte aligned
  uint32_t buckets;

  static __device__ __forceinline__ Mark mark(bool second) { return second ? 0x80000000u : 0x01000000u; }
  // Counts marks: the top bytes of four slots side by side, a counter a byte for each row and for both (at most 255 times four
  // slots: a third of the instructions that shifts and additions slot by slot take, 15 of 109 per 64 windows of a pair of 2 KB).
  struct Count {
    uint32_t in1 = 0, in2 = 0, both = 0;
    __device__ __forceinline__ void add(uint4 v)
    {
      constexpr uint32_t kOnes = 0x01010101u;
      uint32_t const a = __builtin_amdgcn_perm(v.y, v.x, 0x0C0C0703u) | __builtin_amdgcn_perm(v.w, v.z, 0x07030C0Cu), b = a >> 7;
      in1 += a & kOnes;
      in2 += b & kOnes;
      both += a & b & kOnes;
    }
    __device__ __forceinline__ void get(uint32_t (&u)[3]) const
    {
      u[0] = __builtin_amdgcn_sad_u8(in1, 0u, 0u);
      u[1] = __builtin_amdgcn_sad_u8(in2, 0u, 0u);
      u[2] = __builtin_amdgcn_sad_u8(both, 0u, 0u);
    }
  };

  __device__ __forceinline__ uint32_t* at(uint32_t offset) const { return reinterpret_cast<uint32_t*>(reinterpret_cast<uint8_t*>(slots) + offset); }
  // left: a bit a lane.
  template <int N>
  __device__ __forceinline__ void place_at(uint64_t (&left)[N], const uint32_t (&value)[N], const uint32_t (&bucket)[N], const uint32_t (&distance)[N], Mark mark,
                                           uint64_t (&taken)[N]) const
  {
    uint4 v[N];
    uint32_t id[N], s[N], old[N];
    uint64_t tried[N];
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = reinterpret_cast<const uint4*>(slots)[bucket[k]];
    __builtin_amdgcn_sched_barrier(0);  // (all reads on their way before the first is waited for)
#pragma unroll
    for (int k = 0; k < N; ++k) {
      id[k] = (value[k] & kValue) | distance[k] << kDistanceAt;
      // 1 as long as the slots so far hold other values (0 where one is empty or holds this one)
      uint32_t const a0 = least(1u, v[k].x, (v[k].x ^ id[k]) & kSame);
      uint32_t const a1 = least(a0, v[k].y, (v[k].y ^ id[k]) & kSame);
      uint32_t const a2 = least(a1, v[k].z, (v[k].z ^ id[k]) & kSame);
      s[k]              = 16u * bucket[k] + 4u * (a0 + a1 + a2);
      asm("" : "+v"(s[k]));  // (one address for both atomics)
      taken[k]          = ballot64(least(a2, v[k].w, (v[k].w ^ id[k]) & kSame) != 0u);
      tried[k]          = left[k] & ~taken[k];
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
      asm("" : "=v"(old[k]));  // (of the lanes that try nothing it does not matter)
      // (also where the slot holds the value already: cheaper than telling the two apart first)
      if (__builtin_amdgcn_inverse_ballot_w64(tried[k])) old[k] = atomicCAS(at(s[k]), 0u, id[k] | mark);
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
      uint64_t const there = tried[k] & ballot64(((old[k] ^ id[k]) & kSame) == 0u);
      if (__builtin_amdgcn_inverse_ballot_w64(there)) atomicOr(at(s[k]), mark);
      left[k] &= ~(there | (tried[k] & ballot64(old[k] == 0u)));  // (else another value came first)
    }
  }
  __device__ __forceinline__ uint32_t home(uint32_t value) const { return __umulhi(value, buckets); }
  // Buckets from one that is full to the next to be looked at: an odd number up to 31 that the value tells (by bits that a slot
  // holds, so that a slot still tells its home).  With 1 for all the full buckets grow together: at a load of 0.8 the last of 64
  // values put aside had to look at 12 to 15 buckets, now at 6, and the furthest of a pair was 57 from home, now 16.  Random letters,
  // in which no window repeats: 30,000 pairs of 2803-byte rows 1431 -> 820 us, 15,000 of 6100 1565 -> 917, 250,001 of 2 KB words 3515 -> 3490.
  static __device__ __forceinline__ uint32_t step(uint32_t value) { return (value & 15u) * 2u + 1u; }
  // (written out: the compiler makes a comparison and a selection of the minimum with 1)
  static __device__ __forceinline__ uint32_t least(uint32_t a, uint32_t b, uint32_t c)
  {
    uint32_t m;
    asm("v_min3_u32 %0, %1, %2, %3" : "=v"(m) : "v"(a), "v"(b), "v"(c));
    return m;
  }
};

// Whole values, and beside them a bit array for each row: bit s says that the value in slot s occurs there.  Of any size, and
// never full before its last slot is: where a packed set finds no place within kFar buckets (values made for it), and in
// global memory (IN_LDS false), where reads go past the CU's own cache, which does not see what the atomics changed.
template <bool IN_LDS>
__device__ __forceinline__ uint32_t set_word(const uint32_t* p)
{
  if (IN_LDS) return *p;
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool IN_LDS>
struct PlainSet {
  static constexpr uint32_t kFar = 0xFFFFFFFFu;
  using Mark                     = uint32_t*;
  uint32_t* slots;
  uint32_t buckets;
  uint32_t *in1, *in2;

  __device__ __forceinline__ Mark mark(bool second) const { return second ? in2 : in1; }
  __device__ __forceinline__ uint32_t home(uint32_t value) const { return __umulhi(value, buckets); }
  static __device__ __forceinline__ uint32_t step(uint32_t) { return 1u; }  // (every bucket is come by)
  template <int N>
  __device__ __forceinline__ void place_at(uint64_t (&left)[N], const uint32_t (&value)[N], const uint32_t (&bucket)[N], const uint32_t (&)[N], Mark in,
                                           uint64_t (&taken)[N]) const
  {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      bool full = false, in_set = false;
      if (__builtin_amdgcn_inverse_ballot_w64(left[k])) {
        uint32_t s = 4u * bucket[k], v = 0;
        for (int j = 0; j < 4; ++j, ++s) {
          v = set_word<IN_LDS>(&slots[s]);
          if (v == 0u) v = atomicCAS(&slots[s], 0u, value[k]);
          if (v == 0u || v == value[k]) break;
        }
        full = s == 4u * bucket[k] + 4u;
        if (!full) {
          atomicOr(&in[s >> 5], 1u << (s & 31u));
          in_set = true;
        }
      }
      taken[k] = ballot64(full);
      left[k] &= ~ballot64(in_set);
    }
  }
};

// By all lanes: from its home bucket on, until the value is in the set, for the lanes of `left`; what is left found no place.
template <typename Set>
__device__ __forceinline__ uint64_t place(Set const& set, uint64_t left, uint32_t value, typename Set::Mark mark)
{
  uint32_t const values[1] = {value};
  uint32_t bucket[1]       = {set.home(value)}, distance[1] = {0u};
  uint32_t const most      = min(set.buckets, Set::kFar), step = Set::step(value);
  uint64_t lost            = 0;
  while (left != 0) {
    uint64_t l[1] = {left}, taken[1];
    set.template place_at<1>(l, values, bucket, distance, mark, taken);
    left = l[0];
    // on to the next bucket where this one is full (else another value came first: once more, at most until the bucket is full)
    if (__builtin_amdgcn_inverse_ballot_w64(taken[0])) {
      ++distance[0];
      bucket[0] += step;
      if (bucket[0] >= set.buckets) bucket[0] -= set.buckets;
    }
    uint64_t const beyond = left & ballot64(distance[0] >= most);
    lost |= beyond;
    left &= ~beyond;
  }
  return lost;
}

// A share of the hashes by value, for pairs that are cut into parts (other bits than the set's own multiplication uses).  A part
// that its set has no room for is cut in two, as often as it takes (of 2^31 shares none has more than two values): nothing is left over for
// another kernel, so that the host need not wait for the parts (41 pairs of twice 6000 bytes, some of them in parts, 62 -> 49 us).
struct Part {
  uint32_t part, parts;
  // The whole part, then what is left of it: `level` bits of `at` tell which share of it is next.
  uint32_t level = 0, at = 0;
  __device__ __forceinline__ Part share() const { return Part{(part << level) + at, parts << level}; }
  // After a share: whether there is another one.
  __device__ __forceinline__ bool more(bool full)
  {
    if (full) {
      ++level;
      at <<= 1;
      return true;
    }
    ++at;
    while (level != 0 && (at & 1u) == 0) {
      at >>= 1;
      --level;
    }
    return level != 0;
  }
  __device__ __forceinline__ bool holds(uint32_t h) const
  {
    return parts == 1u || __umulhi((h ^ (h >> 15)) * 0x85EBCA6Bu, parts) == part;
  }
};

// A wavefront's own LDS for the tile it hashes.
constexpr uint32_t kLater = 3 * kWave / 2;
struct TileLds {
  alignas(16) uint32_t bytes[kTileWords];
  uint16_t chars[kCharList];
  uint32_t later[kLater];  // hashes that a first look at their bucket did not place
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

// Slots for a pair: room for twice its windows, which are at most its bytes, or what the tier has.
__device__ __forceinline__ uint32_t slots_for(int64_t bytes, uint32_t most)
{
  uint32_t const few = static_cast<uint32_t>(min(bytes, static_cast<int64_t>(most)));
  return min(most, max((2u * few + 63u) / 32u * 32u, PackedSet::kLeast));
}

// ... and in global memory: room for one and a half times its windows.
__device__ __host__ __forceinline__ uint64_t slots_for_global(int64_t bytes)
{
  uint64_t s = 64;
  while (2 * s < 3 * static_cast<uint64_t>(bytes)) s <<= 1;
  return s;
}

// What a set holds for a hash: its product with an odd number (0 for 0, and no two alike).  The compiler does not see what it is,
// or it multiplies once more for the 24 bits that a slot keeps.
__device__ __forceinline__ uint32_t value_of(uint32_t h)
{
  uint32_t v = h * 0x9E3779B1u;
  asm("" : "+v"(v));
  return v;
}

// murmur3_x86_32_unmixed() with seed 0.  Windows in a tile of up to eleven bytes: no loop over their blocks, and every aligned
// dword read once, from one address.
template <int BLOCKS, int N>
__device__ __forceinline__ void few_blocks(WordSrc const (&src)[N], uint32_t len, uint32_t (&h)[N])
{
  auto const mixed = [](uint32_t k) { return rotl32(k * 0xcc9e2d51u, 15) * 0x1b873593u; };
  uint32_t const rem = len & 3u;
  uint32_t words[N][BLOCKS + 2];
#pragma unroll
  for (int i = 0; i < BLOCKS + 2; ++i)
#pragma unroll
    for (int n = 0; n < N; ++n) words[n][i] = src[n].at[i];
  auto const dword = [&](int n, int i) { return __builtin_amdgcn_alignbit(words[n][i + 1], words[n][i], 8u * src[n].mis); };
#pragma unroll
  for (int n = 0; n < N; ++n) h[n] = 0;
#pragma unroll
  for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
    for (int n = 0; n < N; ++n) h[n] = rotl32(h[n] ^ mixed(dword(n, i)), 13) * 5u + 0xe6546b64u;
  if (rem) {
#pragma unroll
    for (int n = 0; n < N; ++n) h[n] ^= mixed(keep_low_bytes(dword(n, BLOCKS), static_cast<int>(rem)));
  }
#pragma unroll
  for (int n = 0; n < N; ++n) h[n] ^= len;
}
template <int N, typename Src>
__device__ __forceinline__ void window_hashes(Src const (&src)[N], uint32_t len, uint32_t (&h)[N])
{
  murmur3_x86_32_unmixed(src, len, 0u, h);
}
template <int N>
__device__ __forceinline__ void window_hashes(WordSrc const (&src)[N], uint32_t len, uint32_t (&h)[N])
{
  // (one length for all windows; what is branched on is told from it anew: the compiler keeps the answers in lanes of vector registers)
  if constexpr (N > 1) asm volatile("" : "+s"(len));
  if (N == 1 || len >= 12)
    murmur3_x86_32_unmixed(src, len, 0u, h);
  else if (len >= 8)
    few_blocks<2>(src, len, h);
  else if (len >= 4)
    few_blocks<1>(src, len, h);
  else
    few_blocks<0>(src, len, h);
}

// A number of wavefronts: known when this is compiled (an int), or a power of two.
struct TeamOf {
  int shift;
  __device__ __forceinline__ operator int() const { return 1 << shift; }
};
__device__ __forceinline__ uint32_t share_of(uint32_t units, int waves) { return units / static_cast<uint32_t>(waves); }
__device__ __forceinline__ uint32_t share_of(uint32_t units, TeamOf waves) { return units >> waves.shift; }

// Hashes the windows of both rows (jaccard.cu:249-292) and inserts the non-zero hashes into the set.  The two rows, one list
// of units of 64 window starts, are shared out evenly among `nwaves` wavefronts, which take up to kTile starts of a row at a
// time.  (Whole tiles in turn left some of four wavefronts a tile more than the others: pairs of 0.8 to 3.3 KB 5 % slower.)
// false: a value found no place.
// FOUR: a lane hashes four windows of a whole tile at a time and not two, so that fewer waits for LDS are left where a SIMD has no more than
// six wavefronts (43,934 pairs of 5.6 to 12.4 KB 1026 -> 978 us; with four wavefronts a pair and seven a SIMD 725 -> 757).
// Nearly every hash finds its place with one look at one bucket, but in most rounds of 64 some lane does not: those are
// put aside and placed 64 at a time, so that a round does not wait for its slowest lane.
template <bool FOUR = false, typename Set, typename Waves>
__device__ __forceinline__ bool insert_pair(ColView const& c1, ColView const& c2, Pair const& pair, int32_t width, Set const& set, Part part, TileLds& lds,
                                            int wave, Waves nwaves, int lane)
{
  auto const hash = [](auto const& src, uint32_t len, auto& h) { window_hashes(src, len, h); };  // jaccard.cu:258: seed 0
  uint64_t lost   = 0;  // (a bit a lane)
  if (static_cast<int64_t>(width) * 4 <= kHalo) {
    int32_t const n1 = static_cast<int32_t>(pair.n1), n2 = static_cast<int32_t>(pair.n2);  // (1.43 GB together at most)
    const uint8_t *const row1 = c1.chars + pair.o1, *const row2 = c2.chars + pair.o2;
    int32_t const units1 = (n1 + kWave - 1) / kWave, units = units1 + (n2 + kWave - 1) / kWave;
    // (22 million units at most, times sixteen)
    int32_t const last   = static_cast<int32_t>(share_of(static_cast<uint32_t>(units) * static_cast<uint32_t>(wave + 1), nwaves));
    uint32_t later = 0, later1 = 0;  // hashes put aside, and how many of them (the first ones) are row 1's: the same in every lane
    bool second    = false;
    auto const place_later = [&] {
      if (!second) later1 = later;
      for (uint32_t i = lane; i - lane < later; i += kWave) {
        bool const have = i < later;
        lost |= place(set, ballot64(have), have ? lds.later[i] : 0u, set.mark(i >= later1));
      }
      later = later1 = 0;
    };
    struct At {
      bool second;
      const uint8_t* row;
      int32_t n, base, end;
      uint32_t cnt;
    };
    auto const tile_at = [&](int32_t unit) {
      At a;
      a.second = unit >= units1;
      a.row    = a.second ? row2 : row1;
      a.n      = a.second ? n2 : n1;
      a.base   = (a.second ? unit - units1 : unit) * kWave;
      a.end    = min(unit + kTile / kWave, a.second ? last : min(last, units1));
      a.cnt    = static_cast<uint32_t>(min((a.end - unit) * kWave, a.n - a.base));
      return a;
    };
    TileBytes tile;  // asked for a tile ahead
    auto const fetch = [&](At const& a) { tile.fetch(a.row + a.base, tile_length(a.n, a.base, a.cnt, width), lane); };
    int32_t const first = static_cast<int32_t>(share_of(static_cast<uint32_t>(units) * static_cast<uint32_t>(wave), nwaves));
    At ahead{};
    if (first < last) {
      ahead = tile_at(first);
      fetch(ahead);
    }
    for (int32_t unit = first; unit < last;) {
      At const a      = ahead;
      second          = a.second;
      auto const mark = set.mark(second);
      unit            = a.end;
      auto const next = [&] {
        if (unit < last) {
          ahead = tile_at(unit);
          fetch(ahead);
        }
      };
      hash_tile_windows<uint32_t, FOUR>(tile, next, a.row, a.n, 0, true, a.base, a.cnt, width, lds.bytes, lds.chars, lane, hash, [&](auto const& valid, auto const& hv) {
        constexpr int N = sizeof(hv) / sizeof(hv[0]);
        uint64_t left[N], taken[N];
        uint32_t value[N], bucket[N], home[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
          left[k]   = ballot64(valid[k]) & ballot64(hv[k] != 0u) & ballot64(part.holds(hv[k]));  // 282-286: zero hashes are dropped
          value[k]  = value_of(hv[k]);
          bucket[k] = set.home(value[k]);
          home[k]   = 0u;
        }
        set.template place_at<N>(left, value, bucket, home, mark, taken);
#pragma unroll
        for (int k = 0; k < N; ++k) {
          if (left[k] != 0) {
            uint32_t const more = static_cast<uint32_t>(__builtin_popcountll(left[k]));
            if (later + more > kLater) place_later();
            if (__builtin_amdgcn_inverse_ballot_w64(left[k])) lds.later[later + lanes_below(left[k])] = value[k];
            later += more;
          }
        }
      });
      if (!second) later1 = later;
      if (later >= kWave) place_later();
    }
    place_later();
    return lost == 0;
  }
  // very wide windows: bytes straight from global memory
#pragma nounroll
  for (int row = 0; row < 2; ++row) {
    const uint8_t* const r = row == 0 ? c1.chars + pair.o1 : c2.chars + pair.o2;
    int64_t const n        = row == 0 ? pair.n1 : pair.n2;
    for (int64_t at = static_cast<int64_t>(wave) * kWave; at < n; at += nwaves * kWave) {
      int64_t const gpos = at + lane, remaining = n - gpos;
      BoundedSrc const src[1] = {{r + gpos, remaining}};
      uint32_t hv[1] = {0u}, hlen;
      if (remaining > 0) {
        uint32_t const readable = static_cast<uint32_t>(min(remaining, static_cast<int64_t>(width) * 4));
        if (window_at(src[0], r + gpos, remaining, readable, gpos == 0, false, width, &hlen)) hash(src, hlen, hv);
      }
      lost |= place(set, ballot64(hv[0] != 0u && part.holds(hv[0])), value_of(hv[0]), set.mark(row != 0));
    }
  }
  return lost == 0;
}

constexpr int kMostWaves = kTierWaves[kTiers - 1];
template <int WAVES>
struct PairScratch {
  TileLds tile[WAVES];
  uint32_t sums[3][WAVES];
  uint32_t full;        // the last pair (counted from 1) whose packed set was full
  uint32_t plain_full;  // whether the plain one was
};

// The sums over a workgroup; what it writes to `scratch` the next pair overwrites behind a barrier of its own.
template <int WAVES>
__device__ __forceinline__ void add_up(uint32_t (&u)[3], PairScratch<WAVES>& scratch, int wave, int lane, uint32_t (&counts)[3])
{
  for (int k = 0; k < 3; ++k) u[k] = wave_inclusive_scan(u[k]);
  if (lane == kWave - 1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) scratch.sums[k][wave] = u[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    counts[k] = 0;
    for (int w = 0; w < WAVES; ++w) counts[k] += scratch.sums[k][w];
  }
}
template <int WAVES, bool IN_LDS>
__device__ __forceinline__ bool count_pair_plain(ColView const& c1, ColView const& c2, Pair const& pair, int32_t width, Part part, PlainSet<IN_LDS> const& set,
                                                 PairScratch<WAVES>& scratch, uint32_t (&counts)[3])
{
  constexpr uint32_t kPairThreads = WAVES * kWave;
  int const lane = lane_id();
  int const wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
  uint32_t const words = set.buckets / 8;  // of bits
  for (uint32_t i = threadIdx.x; i < 4 * set.buckets; i += kPairThreads) set.slots[i] = 0u;
  for (uint32_t i = threadIdx.x; i < words; i += kPairThreads) {
    set.in1[i] = 0u;
    set.in2[i] = 0u;
  }
  if (threadIdx.x == 0) scratch.plain_full = 0u;
  __syncthreads();
  bool const ok = insert_pair(c1, c2, pair, width, set, part, scratch.tile[wave], wave, WAVES, lane);
  if (!ok) scratch.plain_full = 1u;
  __syncthreads();
  uint32_t u[3] = {0, 0, 0};
  for (uint32_t i = threadIdx.x; i < words; i += kPairThreads) {
    uint32_t const a = set_word<IN_LDS>(&set.in1[i]), b = set_word<IN_LDS>(&set.in2[i]);
    u[0] += __builtin_popcount(a);
    u[1] += __builtin_popcount(b);
    u[2] += __builtin_popcount(a & b);
  }
  bool const full = scratch.plain_full != 0u;
  add_up(u, scratch, wave, lane, counts);
  return !full;
}
// The plain set where a packed one of `nslots` slots lies in LDS: sixteen of seventeen of its words are slots, the others the
// bits.  (Room for the windows of the longest pair of a tier all the same: 0.8 * 17 / 16.)
__device__ __forceinline__ PlainSet<true> plain_in(uint32_t* slots, uint32_t nslots)
{
  uint32_t const words = nslots / 34;  // of bits, of a row
  return PlainSet<true>{slots, 8 * words, slots + 32 * words, slots + 33 * words};
}
// What the lanes of a pair's wavefronts counted in a packed set (of fewer than 65,536 slots), two of the three numbers in one; behind a barrier
// the pair's first wavefront adds up.  (All of them added up all three with a read each: 63,333 pairs of twice 6000 bytes 3596 ->
// 3424 us, 200 of twice 200 23.2 -> 21.5.)
template <int W>
__device__ __forceinline__ void put_counts(PackedSet::Count const& in, uint32_t (&sums)[3][W], int wave, int lane)
{
  uint32_t u[3];
  in.get(u);
  uint32_t const both_rows = wave_inclusive_scan(u[0] | u[1] << 16), common = wave_inclusive_scan(u[2]);
  if (lane == kWave - 1) {
    sums[0][wave] = both_rows;
    sums[1][wave] = common;
  }
}
template <int W>
__device__ __forceinline__ void get_counts(const uint32_t (&sums)[3][W], int first, int waves, int lane, uint32_t (&counts)[3])
{
  uint32_t v0 = 0, v1 = 0;
  if (lane < waves) {
    v0 = sums[0][first + lane];
    v1 = sums[1][first + lane];
  }
  v0        = wave_bcast(wave_inclusive_scan(v0), kWave - 1);
  v1        = wave_bcast(wave_inclusive_scan(v1), kWave - 1);
  counts[0] = v0 & 0xFFFFu;
  counts[1] = v0 >> 16;
  counts[2] = v1;
}
// One row pair (or a part of it) by WAVES wavefronts with a set of `nslots` slots (a multiple of 32): inserts both rows, counts,
// and leaves the set empty, as it was before (start_pairs).  `number`: of the pair among the workgroup's, from 1.  The counts are
// thread 0's; false (everywhere) when the set was full.
template <int WAVES>
__device__ __forceinline__ void start_pairs(uint32_t* slots, uint32_t nslots, PairScratch<WAVES>& scratch)
{
  // (the slots are 16-byte aligned: whole uint4 stores)
  for (uint32_t i = threadIdx.x; i < nslots / 4; i += WAVES * kWave) reinterpret_cast<uint4*>(slots)[i] = make_uint4(0u, 0u, 0u, 0u);
  if (threadIdx.x == 0) scratch.full = 0u;
  __syncthreads();
}
template <int WAVES>
__device__ __forceinline__ bool count_pair(ColView const& c1, ColView const& c2, Pair const& pair, int32_t width, Part part, uint32_t* slots, uint32_t nslots,
                                           PairScratch<WAVES>& scratch, uint32_t number, uint32_t (&counts)[3])
{
  int const lane = lane_id();
  int const wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
  bool const ok  = insert_pair<(WAVES >= 12)>(c1, c2, pair, width, PackedSet{slots, nslots / 4}, part, scratch.tile[wave], wave, WAVES, lane);
  if (!ok) scratch.full = number;
  __syncthreads();
  bool const full = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(scratch.full))) == number;
  PackedSet::Count in;
  for (uint32_t i = threadIdx.x; i < nslots / 4; i += WAVES * kWave) {
    uint4* const four = reinterpret_cast<uint4*>(slots) + i;
    in.add(*four);
    *four = make_uint4(0u, 0u, 0u, 0u);
  }
  put_counts(in, scratch.sums, wave, lane);
  __syncthreads();
  if (wave == 0) get_counts(scratch.sums, 0, WAVES, lane, counts);
  return !full;
}
// A pair that found its packed set full is marked in its list, and done once more with a plain set when the workgroup is through
// with the others (not right away: the registers that takes are then not taken from the usual case).
constexpr uint32_t kOnceMore = 0x80000000u;  // (rows are fewer)

// Work lists in `work`: a header -- [i] = pairs on list i, [kLists] = null rows of the result,
// [8..9] = the most bytes a pair of the global list has (64 bits), [kTotalParts] = parts of all pairs on the list of pairs in parts,
// and, on a cache line that nobody reads (63,333 pairs of twice 6000 bytes 3348 -> 3246 us), pieces of work handed out by each of
// the two kernels that hand some out ([kNextPiece], [kNextPart]: where there are more than kMostParts parts both of them run) -- then
// four counters (|A|, |B|, |A n B|, parts done) for
// every entry of the list of pairs in parts, `rows` entries for each list, and the first kMostParts of the parts themselves
// (a pair's entry | its number << 27, and the pair).
constexpr int kListHeader = 64;
constexpr int kToldWords  = 16;  // of the header, that the host is told
constexpr int kMostBytes  = 8;
constexpr int kTotalParts = 10;
constexpr int kNextPiece  = 32;  // jaccard_teams_kernel
constexpr int kNextPart   = 48;  // jaccard_parts_kernel
constexpr int32_t kLookRows = 131072;  // see nvtext_amd_jaccard_index
constexpr uint32_t kMostParts = 1u << 16;  // (of pairs of 0.8 GB and more)
static_assert(kMostParts <= 1u << 27 && kMaxParts <= 32);
__host__ __device__ __forceinline__ uint32_t most_parts(int64_t rows)
{
  return rows < kMostParts / kMaxParts ? static_cast<uint32_t>(rows * kMaxParts) : kMostParts;
}
__host__ __device__ __forceinline__ size_t work_words(int64_t rows) { return kListHeader + static_cast<size_t>(kLists + 4) * static_cast<size_t>(rows) + 2 * static_cast<size_t>(most_parts(rows)); }
__device__ __forceinline__ uint32_t* list_entries(uint32_t* work, int list, int64_t rows) { return work + kListHeader + (4 + list) * rows; }
__device__ __forceinline__ uint32_t* part_counters(uint32_t* work) { return work + kListHeader; }
// (the lists are an even number of words: 8-byte records, aligned)
static_assert((kLists + 4) % 2 == 0);
__device__ __forceinline__ uint2* single_parts(uint32_t* work, int64_t rows) { return reinterpret_cast<uint2*>(work + kListHeader + (kLists + 4) * rows); }
struct WaveSetLds {
  alignas(16) uint32_t slots[kSlots[0]];
  TileLds tile;
};
static_assert(kSlots[0] == PackedSet::kLeast, "every pair of a wavefront takes all slots");

// A workgroup sizes `per_group` consecutive pairs at once (at most kThreads: threads <-> pairs, coalesced offset loads),
// lists those that need more than a wavefront's own set for the later kernels with one atomic per list (atomics on one
// cache line run at about 150 M/s: one per wavefront and list was most of this kernel's time), and its wavefronts do the
// others, each taking the next one when it is done with one.  A column of few pairs is shared out over more workgroups.
// told.arrivals (a column of up to kLookRows pairs): the first workgroups list 256 pairs each before they do their own, in counters
// there, and the one that is last to have done so tells the host the header, while all have their own pairs yet to do.  (Were every
// workgroup to list its own, of which there are 1,000 to 2,000 for the sake of those pairs, their atomics would be all of the
// time: 3,333 pairs of twice 6000 bytes took 24 us to list, now 14, and 8,166 42, now 17; 7,500 of twice 200 bytes 36, now 24.)
struct Told {
  Arrivals* arrivals;
  uint32_t listers;
  uint32_t* host;
  HostPost post;
};
__global__ void __launch_bounds__(kThreads) jaccard_wave_kernel(ColView c1, ColView c2, int32_t width, float* __restrict__ out,
                                                                uint32_t* __restrict__ work, int per_group, Told told)
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
  auto const empty_set = [&] {
    for (uint32_t i = lane; i < kSlots[0] / 4; i += kWave) reinterpret_cast<uint4*>(lds.slots)[i] = make_uint4(0u, 0u, 0u, 0u);
    wave_sync();
  };
  // lists the pairs r of this workgroup's threads in `counts`
  auto const list_pairs = [&](bool later, int64_t r, int64_t bytes, uint32_t* counts) {
    int const list = list_of(bytes);
    uint32_t at    = 0;
    if (later) at = atomicAdd(&listed[list], 1u);
    __syncthreads();
    if (threadIdx.x < kLists && listed[threadIdx.x] != 0u) place[threadIdx.x] = atomicAdd(&counts[threadIdx.x], listed[threadIdx.x]);
    __syncthreads();
    if (!later) return;
    at += place[list];
    list_entries(work, list, rows)[at] = static_cast<uint32_t>(r);
    if (list == kPartsList) {
      reinterpret_cast<uint4*>(part_counters(work))[at] = make_uint4(0u, 0u, 0u, 0u);
      uint32_t const parts = static_cast<uint32_t>(parts_of(bytes)), first = atomicAdd(&counts[kTotalParts], parts);
      for (uint32_t p = 0; p < parts && first + p < most_parts(rows); ++p) single_parts(work, rows)[first + p] = make_uint2(at | p << 27, static_cast<uint32_t>(r));
    }
    if (list == kGlobalList) atomicMax(reinterpret_cast<unsigned long long*>(&counts[kMostBytes]), static_cast<unsigned long long>(bytes));
  };
  if (told.arrivals && blockIdx.x < told.listers) {
    if (threadIdx.x < kLists) listed[threadIdx.x] = 0u;
    __syncthreads();
    int64_t const r     = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    int64_t const bytes = r < rows ? pair_at(c1, c2, r).bytes() : 0;
    list_pairs(bytes > most_bytes(kSlots[0]), r, bytes, told.arrivals->words);
    __threadfence();  // (all that was added is there before this workgroup is seen to have arrived)
    __syncthreads();
    if (wave == 0) {
      uint32_t last = 0;
      if (lane == 0) last = atomicAdd(&told.arrivals->sum, 1ull) + 1ull == told.listers;
      if (wave_bcast(last, 0) != 0) {
        // (all is left as it was found: zeros)
        if (lane == 0) atomicExch(&told.arrivals->sum, 0ull);
        uint32_t v = 0;
        if (lane < kToldWords) {
          v               = atomicExch(&told.arrivals->words[lane], 0u);
          told.host[lane] = v;
        }
        if (lane < kListHeader) work[lane] = v;
        __threadfence_system();
        if (lane == 0) told.post.send();
      }
    }
  }
  for (int64_t base = static_cast<int64_t>(blockIdx.x) * per_group; base < rows; base += static_cast<int64_t>(gridDim.x) * per_group) {
    __syncthreads();
    if (threadIdx.x < kLists) listed[threadIdx.x] = 0u;
    if (threadIdx.x == 0) solos = next = 0u;
    __syncthreads();
    int64_t const r   = base + threadIdx.x;
    bool const have   = r < rows && static_cast<int>(threadIdx.x) < per_group;
    int64_t const all = have ? pair_at(c1, c2, r).bytes() : 0;
    bool const later  = have && all > most_bytes(kSlots[0]);
    if (have && !later) solo[atomicAdd(&solos, 1u)] = static_cast<uint32_t>(r);
    if (told.arrivals)
      __syncthreads();
    else
      list_pairs(later, r, all, work);
    bool again = false;
    if (solos != 0) empty_set();  // (and every pair leaves it so: 1,900,000 pairs of twice 200 bytes 2789 -> 2737 us)
    for (;;) {
      uint32_t t = 0;
      if (lane == 0) t = atomicAdd(&next, 1u);
      t = wave_bcast(t, 0);
      if (t >= solos) break;
      uint32_t const pr = solo[t];
      Pair const q      = uniform_pair_at(c1, c2, pr);
      bool const ok = insert_pair(c1, c2, q, width, PackedSet{lds.slots, kSlots[0] / 4}, Part{0, 1}, lds.tile, 0, 1, lane);
      wave_sync();
      if (ballot64(!ok) != 0) {
        empty_set();
        if (lane == 0) solo[t] = pr | kOnceMore;
        again = true;
        continue;
      }
      PackedSet::Count in;
      uint32_t u[3];
#pragma unroll
      for (uint32_t i = lane; i < kSlots[0] / 4; i += kWave) {
        uint4* const four = reinterpret_cast<uint4*>(lds.slots) + i;
        in.add(*four);
        *four = make_uint4(0u, 0u, 0u, 0u);
      }
      in.get(u);
      uint32_t const u1 = wave_inclusive_scan(u[0] | u[1] << 16);  // (at most 1024 in either half)
      u[2]              = wave_inclusive_scan(u[2]);
      if (lane == kWave - 1) out[pr] = index_of(u1 & 0xFFFFu, u1 >> 16, u[2]);
      wave_sync();
    }
    if (!again) continue;
    // what was marked so far: this wavefront's own at least
    for (uint32_t t = 0; t < solos; ++t) {
      wave_sync();
      uint32_t const pr = solo[t] & ~kOnceMore;
      uint32_t first    = 0;
      if (lane == 0) first = atomicAnd(&solo[t], ~kOnceMore);  // (one of the wavefronts takes it)
      if ((wave_bcast(first, 0) & kOnceMore) == 0u) continue;
      for (uint32_t i = lane; i < kSlots[0]; i += kWave) lds.slots[i] = 0u;
      wave_sync();
      PlainSet<true> const plain = plain_in(lds.slots, kSlots[0]);
      insert_pair(c1, c2, uniform_pair_at(c1, c2, pr), width, plain, Part{0, 1}, lds.tile, 0, 1, lane);
      wave_sync();
      uint32_t u[3] = {0, 0, 0};
      for (uint32_t i = lane; i < plain.buckets / 8; i += kWave) {
        u[0] += __builtin_popcount(plain.in1[i]);
        u[1] += __builtin_popcount(plain.in2[i]);
        u[2] += __builtin_popcount(plain.in1[i] & plain.in2[i]);
      }
      for (uint32_t& x : u) x = wave_inclusive_scan(x);
      if (lane == kWave - 1) out[pr] = index_of(u[0], u[1], u[2]);
    }
  }
}

// The pairs of a tier's list, one workgroup of WAVES wavefronts and one set of SLOTS slots per pair.
template <int TIER>
__global__ void __launch_bounds__(kTierWaves[TIER] * kWave, kSimdWaves[TIER]) jaccard_listed_kernel(ColView c1, ColView c2, int32_t width, float* __restrict__ out,
                                                                                  uint32_t* __restrict__ work)
{
  constexpr uint32_t SLOTS = kSlots[TIER];
  constexpr int WAVES      = kTierWaves[TIER];
  __shared__ alignas(16) uint32_t slots[SLOTS];
  __shared__ PairScratch<WAVES> scratch;
  int64_t const rows   = c1.size;
  uint32_t const count = work[TIER - 1];
  if (blockIdx.x >= count) return;
  uint32_t* const entries = list_entries(work, TIER - 1, rows);
  start_pairs(slots, SLOTS, scratch);
  uint32_t number = 0;
  bool again      = false;
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    uint32_t const r = entries[i];
    Pair const pair  = uniform_pair_at(c1, c2, r);
    uint32_t counts[3];
    bool const ok = count_pair<WAVES>(c1, c2, pair, width, Part{0, 1}, slots, slots_for(pair.bytes(), SLOTS), scratch, ++number, counts);
    if (!ok) {
      again = true;
      if (threadIdx.x == 0) entries[i] = r | kOnceMore;
    } else if (threadIdx.x == 0) {
      out[r] = index_of(counts[0], counts[1], counts[2]);
    }
  }
  if (!again) return;
  __syncthreads();  // (what thread 0 wrote is there)
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    uint32_t const r = *const_cast<volatile uint32_t*>(&entries[i]);
    if ((r & kOnceMore) == 0u) continue;
    uint32_t counts[3];
    count_pair_plain<WAVES>(c1, c2, uniform_pair_at(c1, c2, r & ~kOnceMore), width, Part{0, 1}, plain_in(slots, SLOTS), scratch, counts);
    if (threadIdx.x == 0) out[r & ~kOnceMore] = index_of(counts[0], counts[1], counts[2]);
    __syncthreads();
  }
}

// By one thread: adds the counts of a part of pair r, which has this entry of its list.  The last part to be done writes the index.
__device__ __forceinline__ void finish_part(uint32_t* work, uint32_t r, uint32_t entry, uint32_t parts, uint32_t const (&counts)[3], float* out)
{
  uint32_t* const at = part_counters(work) + 4 * static_cast<int64_t>(entry);
  for (int k = 0; k < 3; ++k) atomicAdd(&at[k], counts[k]);
  __threadfence();
  if (atomicAdd(&at[3], 1u) + 1u == parts) {
    __threadfence();
    out[r] = index_of(atomicAdd(&at[0], 0u), atomicAdd(&at[1], 0u), atomicAdd(&at[2], 0u));
  }
}
// The pairs in parts of a column whose lists the host does not look at, or where they have more than kMostParts: then all that the
// pairs could have are gone through.
constexpr int kPartsTier = kTiers - 1;
__global__ void __launch_bounds__(kTierWaves[kPartsTier] * kWave) jaccard_parts_kernel(ColView c1, ColView c2, int32_t width, float* __restrict__ out,
                                                                                       uint32_t* __restrict__ work)
{
  constexpr uint32_t SLOTS = kSlots[kPartsTier];
  constexpr int WAVES      = kTierWaves[kPartsTier];
  __shared__ alignas(16) uint32_t slots[SLOTS];
  __shared__ PairScratch<WAVES> scratch;
  __shared__ uint32_t next;
  int64_t const rows    = c1.size;
  bool const known      = work[kTotalParts] <= most_parts(rows);
  uint64_t const pieces = known ? work[kTotalParts] : static_cast<uint64_t>(work[kPartsList]) * kMaxParts;
  if (blockIdx.x >= pieces) return;
  start_pairs(slots, SLOTS, scratch);
  uint32_t number = 0;
  for (uint32_t piece = blockIdx.x; piece < pieces;) {
    uint32_t ahead = 0;
    if (threadIdx.x == 0) ahead = atomicAdd(&work[kNextPart], 1u) + gridDim.x;
    uint2 const e    = known ? single_parts(work, rows)[piece] : make_uint2(0u, 0u);
    uint32_t const i = known ? e.x & 0x07FFFFFFu : piece / kMaxParts;
    uint32_t const r = known ? e.y : list_entries(work, kPartsList, rows)[i];
    Pair const pair  = uniform_pair_at(c1, c2, r);
    Part part{known ? e.x >> 27 : piece % static_cast<uint32_t>(kMaxParts), static_cast<uint32_t>(parts_of(pair.bytes()))};
    if (part.part < part.parts) {
      uint32_t sum[3] = {0, 0, 0};
      for (bool more = true; more;) {
        uint32_t counts[3];
        bool const ok = count_pair<WAVES>(c1, c2, pair, width, part.share(), slots, SLOTS, scratch, ++number, counts);
        if (ok)
          for (int k = 0; k < 3; ++k) sum[k] += counts[k];
        more = part.more(!ok);
      }
      if (threadIdx.x == 0) finish_part(work, r, i, part.parts, sum, out);
    }
    if (threadIdx.x == 0) next = ahead;
    __syncthreads();
    piece = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(next)));
    __syncthreads();
  }
}

// All lists but the last in one launch, where the host knows what is on them (columns of up to kLookRows pairs).  With a launch a
// tier each waits for its slowest pair before the next begins.  A workgroup of sixteen wavefronts and the largest set takes
// pieces of work until none is left: a part of a pair, a pair of the last two tiers, two pairs of tier 2 or four of tier 1,
// each by a team of its wavefronts with its share of the set; the longest first.  The teams share the barriers.  Pairs of twice 1500
// bytes on average, lengths lognormal (0.8), with the first three tiers' own kernels and in this launch: 166 of them 59 and 27 us, 466 60 and 28,
// 2,000 72 and 48; of twice 6000, 1,666 200 and 156; 7,500 of twice 200 41 and 35.  What bounds it is one piece: its bytes are hashed
// by one CU.
// With more than kTeamPieces pieces of the first three tiers these have their own kernels, more of whose wavefronts fit a CU (13,333
// pairs of twice 1500 bytes 176 us with their own kernels and 205 in this launch, 32,666 341 and 469, 16,666 of twice 6000 868 and 945; between
// them it depends on the lengths: 3,333 of twice 6000 219 and 188).
struct Pieces {
  uint32_t parts, tier4, tier3, tier2, tier1;  // where the pieces of each kind end
  uint32_t pairs2, pairs1;                     // of the last two kinds
  int shift2, shift1;                          // wavefronts of a team of these, their logarithm
};
constexpr uint32_t kTeamPieces = 1536;  // of the first three tiers at most
constexpr int kTeamWaves       = kMostWaves;
constexpr int kTeamShift       = 4;
static_assert(kTeamWaves == 1 << kTeamShift);
constexpr uint32_t kTeamSlots  = kSlots[kTiers - 1];
struct TeamScratch {
  TileLds tile[kTeamWaves];
  uint32_t sums[3][kMostWaves];
  uint32_t full[kTeamWaves];  // of a team's first wavefront: the set was full
  uint32_t next;
};
__global__ void __launch_bounds__(kTeamWaves * kWave) jaccard_teams_kernel(ColView c1, ColView c2, int32_t width, float* __restrict__ out,
                                                                           uint32_t* __restrict__ work, Pieces pieces)
{
  __shared__ alignas(16) uint32_t slots[kTeamSlots];
  __shared__ TeamScratch scratch;
  int64_t const rows = c1.size;
  int const lane     = lane_id();
  int const wave     = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
  for (uint32_t i = threadIdx.x; i < kTeamSlots / 4; i += kTeamWaves * kWave) reinterpret_cast<uint4*>(slots)[i] = make_uint4(0u, 0u, 0u, 0u);
  bool const more = pieces.tier1 > gridDim.x;
  for (uint32_t piece = blockIdx.x; piece < pieces.tier1;) {
    // the team's wavefronts, its share of the set, and the entry of its list that it has (none: `have` is false)
    int shift = kTeamShift, list = kPartsList;
    uint32_t most = kTeamSlots, entry = piece;
    bool have     = true;
    if (piece >= pieces.tier2) {
      shift = pieces.shift1, list = 0, most = kSlots[1];
      entry = ((piece - pieces.tier2) << (kTeamShift - shift)) + (static_cast<uint32_t>(wave) >> shift);
      have  = entry < pieces.pairs1;
    } else if (piece >= pieces.tier3) {
      shift = pieces.shift2, list = 1, most = kSlots[2];
      entry = ((piece - pieces.tier3) << (kTeamShift - shift)) + (static_cast<uint32_t>(wave) >> shift);
      have  = entry < pieces.pairs2;
    } else if (piece >= pieces.tier4) {
      list = 2, most = kSlots[3], entry = piece - pieces.tier4;
    } else if (piece >= pieces.parts) {
      list = 3, entry = piece - pieces.parts;
    }
    TeamOf const waves{shift};
    int const team      = wave >> shift, own = wave & (waves - 1);
    uint32_t* const set = slots + static_cast<uint32_t>(team) * most;
    Part part{0, 1};
    uint32_t counter = 0, r = 0;
    if (list == kPartsList) {
      uint2 const e = single_parts(work, rows)[piece];
      counter       = e.x & 0x07FFFFFFu;
      part.part     = e.x >> 27;
      r             = e.y;
    } else if (have) {
      r = list_entries(work, list, rows)[entry];
    }
    r = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(r)));
    Pair pair{0, 0, 0, 0};
    if (have) pair = uniform_pair_at(c1, c2, r);
    if (list == kPartsList) part.parts = static_cast<uint32_t>(parts_of(pair.bytes()));
    uint32_t const nslots = list == kPartsList ? most : slots_for(pair.bytes(), most);
    uint32_t next = pieces.tier1;
    if (more && threadIdx.x == 0) next = atomicAdd(&work[kNextPiece], 1u) + gridDim.x;
    uint32_t total[3], sum[3] = {0, 0, 0};
    bool full, any;
    for (;;) {
      if (lane == 0) scratch.full[wave] = 0u;
      __syncthreads();  // (the set is empty, the flags are down, the sums of the piece before have been read)
      bool const ok = insert_pair<true>(c1, c2, pair, width, PackedSet{set, nslots / 4}, part.share(), scratch.tile[wave], own, waves, lane);
      if (!ok) scratch.full[wave - own] = 1u;
      if (threadIdx.x == 0) scratch.next = next;
      __syncthreads();
      uint32_t const flag = lane < kTeamWaves ? scratch.full[lane] : 0u;
      full                = wave_bcast(flag, wave - own) != 0;
      any                 = ballot64(flag != 0) != 0;
      PackedSet::Count in;
      for (uint32_t i = own * kWave + lane; i < nslots / 4; i += waves * kWave) {
        uint4* const four = reinterpret_cast<uint4*>(set) + i;
        in.add(*four);
        *four = make_uint4(0u, 0u, 0u, 0u);
      }
      put_counts(in, scratch.sums, wave, lane);
      __syncthreads();
      if (own == 0) get_counts(scratch.sums, wave, waves, lane, total);
      if (list != kPartsList) break;
      if (!full)
        for (int k = 0; k < 3; ++k) sum[k] += total[k];
      if (!part.more(full)) break;
    }
    next = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(scratch.next)));
    if (list != kPartsList && any) {
      // a value found no place in a packed set (none in text): such a pair once more with a plain one; every team comes along
      PlainSet<true> const plain = plain_in(set, most);
      Pair const again           = full ? pair : Pair{0, 0, 0, 0};
      uint32_t const words       = plain.buckets / 8;
      for (uint32_t i = own * kWave + lane; i < most; i += waves * kWave) set[i] = 0u;
      __syncthreads();
      insert_pair(c1, c2, again, width, plain, part, scratch.tile[wave], own, waves, lane);
      __syncthreads();
      uint32_t u[3] = {0, 0, 0};
      for (uint32_t i = own * kWave + lane; i < words; i += waves * kWave) {
        u[0] += __builtin_popcount(plain.in1[i]);
        u[1] += __builtin_popcount(plain.in2[i]);
        u[2] += __builtin_popcount(plain.in1[i] & plain.in2[i]);
      }
      for (int k = 0; k < 3; ++k) u[k] = wave_inclusive_scan(u[k]);
      if (lane == kWave - 1)
        for (int k = 0; k < 3; ++k) scratch.sums[k][wave] = u[k];
      __syncthreads();
      if (full) {
        for (int k = 0; k < 3; ++k) {
          total[k] = 0;
          for (int w = 0; w < waves; ++w) total[k] += scratch.sums[k][wave - own + w];
        }
      }
      for (uint32_t i = own * kWave + lane; i < most; i += waves * kWave) set[i] = 0u;
    }
    if (have && own == 0 && lane == 0) {
      if (list != kPartsList)
        out[r] = index_of(total[0], total[1], total[2]);
      else
        finish_part(work, r, counter, part.parts, sum, out);
    }
    piece = next;
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
    count_pair_plain<kWaves, false>(c1, c2, pair, width, Part{0, 1}, PlainSet<false>{mine, need / 4, mine + table_slots, mine + table_slots + table_slots / 32},
                                    scratch, counts);
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
  // In a column of few pairs the launches of the other kernels, most of which would find their lists empty, are more than
  // the work: the host looks at the lists first and launches what has something to do (35,000 pairs of twice 200 bytes 148 -> 127 us,
  // 100,000 278 -> 264).  In a larger one its wait and the listing before all else cost more (245,000 527 -> 554, 250,001 of
  // twice 2 KB 3500 -> 3605).
  uint64_t* const pinned = host_scalars();
  CallArrivals const arrivals(mr, rows <= kLookRows && pinned);
  Arrivals* const own    = arrivals.get();
  bool const look        = own != nullptr;
  if (!own) launch_fill_u32(lists, 0u, kListHeader, stream);

  ColView const v1 = make_view(*input1);
  ColView const v2 = make_view(*input2);
  float* const values = static_cast<float*>(out->data);
  int const cus       = device_cus();
  if (with_mask) {
    int32_t const words = (rows + 31) / 32;
    hipLaunchKernelGGL(and_bitmask_kernel, dim3((words + 255) / 256), dim3(256), 0, stream, out->null_mask,
                       input1->null_count > 0 ? input1->null_mask : nullptr, input1->offset,
                       input2->null_count > 0 ? input2->null_mask : nullptr, input2->offset, rows, words, own ? &own->words[kLists] : &lists[kLists]);
  }
  Told told{own, static_cast<uint32_t>((static_cast<int64_t>(rows) + kThreads - 1) / kThreads), reinterpret_cast<uint32_t*>(pinned), HostPost{}};
  if (own) told.post = new_post();
  {
    ProfileScope ps("jaccard_wave_kernel", stream);
    int per_group = kThreads;
    while (per_group > kWaves && rows / per_group < 4 * cus) per_group /= 2;
    int64_t const groups = (static_cast<int64_t>(rows) + per_group - 1) / per_group;
    unsigned const grid  = static_cast<unsigned>(std::min<int64_t>(groups, static_cast<int64_t>(cus) * 64));
    hipLaunchKernelGGL(jaccard_wave_kernel, dim3(grid), dim3(kThreads), 0, stream, v1, v2, width, values, lists, per_group, told);
  }
  // what the host has to know: the header of the lists
  uint32_t copied[kToldWords] = {};
  const uint32_t* const head   = pinned ? reinterpret_cast<const uint32_t*>(pinned) : copied;
  auto const read_header       = [&]() -> hipError_t {
    if (!pinned) {
      hipError_t const e = hipMemcpyAsync(copied, lists, sizeof(copied), hipMemcpyDeviceToHost, stream);
      return e == hipSuccess ? hipStreamSynchronize(stream) : e;
    }
    HostPost const post = new_post();
    hipLaunchKernelGGL(publish_header_kernel, dim3(1), dim3(kToldWords), 0, stream, lists, reinterpret_cast<uint32_t*>(pinned), post);
    hipError_t const e = hipGetLastError();
    return e == hipSuccess ? wait_for_post(post, stream) : e;
  };
  hipError_t e = hipGetLastError();
  if (look) {
    if (e == hipSuccess) e = wait_for_post(told.post, stream);
    if (e != hipSuccess) arrivals.failed();  // (nobody knows what it holds)
  }
  auto const listed = [&](int list) { return look ? static_cast<int32_t>(head[list]) : rows; };
  auto const grid_of = [&](int list, int per_cu) { return dim3(static_cast<unsigned>(std::min<int64_t>(listed(list), static_cast<int64_t>(cus) * per_cu))); };
  bool few = false;  // pairs on the first three lists
  bool in_pieces = false;  // the pairs in parts
  Pieces pieces{};
  if (look && e == hipSuccess) {
    in_pieces    = head[kTotalParts] <= most_parts(rows);
    pieces.parts = in_pieces ? head[kTotalParts] : 0u;
    pieces.tier4 = pieces.parts + static_cast<uint32_t>(listed(3));
    // (fewer pieces than CUs: a workgroup for every pair)
    uint32_t const pairs = static_cast<uint32_t>(listed(2)) + static_cast<uint32_t>(listed(1)) + static_cast<uint32_t>(listed(0));
    bool const alone     = pieces.tier4 + pairs <= static_cast<uint32_t>(cus);
    static_assert(kTierWaves[2] == 8 && kTierWaves[1] == 4);
    pieces.shift2        = alone ? kTeamShift : 3;
    pieces.shift1        = alone ? kTeamShift : 2;
    pieces.pairs2        = static_cast<uint32_t>(listed(1));
    pieces.pairs1        = static_cast<uint32_t>(listed(0));
    auto const teams_of  = [](uint32_t pairs, int shift) { return (pairs + (1u << (kTeamShift - shift)) - 1u) >> (kTeamShift - shift); };
    uint32_t const n3 = static_cast<uint32_t>(listed(2)), n2 = teams_of(pieces.pairs2, pieces.shift2), n1 = teams_of(pieces.pairs1, pieces.shift1);
    few          = n3 + n2 + n1 <= kTeamPieces;
    pieces.tier3 = pieces.tier4 + (few ? n3 : 0u);
    pieces.tier2 = pieces.tier3 + (few ? n2 : 0u);
    pieces.tier1 = pieces.tier2 + (few ? n1 : 0u);
    if (pieces.tier1 > 0) {
      ProfileScope ps("jaccard_teams_kernel", stream);
      hipLaunchKernelGGL(jaccard_teams_kernel, dim3(std::min<uint32_t>(pieces.tier1, static_cast<uint32_t>(cus))), dim3(kTeamWaves * kWave), 0, stream, v1, v2,
                         width, values, lists, pieces);
    }
  }
  if (!few && e == hipSuccess && listed(0) > 0) {
    ProfileScope ps("jaccard_listed_kernel<1>", stream);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(jaccard_listed_kernel<1>), grid_of(0, 28), dim3(kTierWaves[1] * kWave), 0, stream, v1, v2, width, values, lists);
  }
  if (!few && e == hipSuccess && listed(1) > 0) {
    ProfileScope ps("jaccard_listed_kernel<2>", stream);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(jaccard_listed_kernel<2>), grid_of(1, 12), dim3(kTierWaves[2] * kWave), 0, stream, v1, v2, width, values, lists);
  }
  if (!few && e == hipSuccess && listed(2) > 0) {
    ProfileScope ps("jaccard_listed_kernel<3>", stream);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(jaccard_listed_kernel<3>), grid_of(2, 8), dim3(kTierWaves[3] * kWave), 0, stream, v1, v2, width, values, lists);
  }
  if (!look && e == hipSuccess) {
    ProfileScope ps("jaccard_listed_kernel<4>", stream);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(jaccard_listed_kernel<4>), grid_of(3, 4), dim3(kTierWaves[4] * kWave), 0, stream, v1, v2, width, values, lists);
  }
  if (!in_pieces && e == hipSuccess) {
    ProfileScope ps("jaccard_parts_kernel", stream);
    hipLaunchKernelGGL(jaccard_parts_kernel, dim3(static_cast<unsigned>(cus)), dim3(kTierWaves[kPartsTier] * kWave), 0, stream,
                       v1, v2, width, values, lists);
  }
  if (e == hipSuccess && !look) e = read_header();
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
