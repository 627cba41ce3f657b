// nvtext::normalize_characters for gfx950: the BERT basic-tokenizer clean-up of a strings column
// (cpp/src/text/normalize.cu:219-573).
//
// The reference expands every input byte into three uint32 slots in global memory, fixes the special tokens up
// in a second kernel, reduces the slots to row sizes and compacts them.  Here a workgroup (in a large column a
// wavefront) takes a tile of 2048 input bytes, plus a few either side, eight consecutive bytes to a lane,
// and the column is walked twice: once to learn how many bytes each tile produces, once to write them,
// coalesced, at the offsets a scan of those counts gives.  HBM sees the input twice and the output once; the
// slots never leave the CU.
#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "common.cuh"

struct nvtext_amd_character_normalizer {
  int device            = 0;
  int32_t do_lower      = 0;
  uint32_t* ascii       = nullptr;  // device, 256: slot 0 | slot 1 << 8 | slot 2 << 16 | bytes << 24 of the code points below 0x80, zeros
  uint4* bmp            = nullptr;  // device, 65536: {slot 0, slot 1, slot 2, bytes} of the code points below 0x10000, and 65536 of their strings
  uint8_t* sizes        = nullptr;  // device, 65536: the bytes alone
  uint32_t* entries     = nullptr;  // device, kCodepoints: category << 24 | multi << 23 | replacement
  uint64_t* second      = nullptr;  // device, kCodepoints: second << 32 | third replacement code point
  uint8_t* token_chars  = nullptr;  // device: the special tokens, sorted then lower-cased
  int32_t* token_offset = nullptr;  // device, tokens + 1
  int32_t tokens        = 0;
  nvtext_amd::DeviceStore store;    // all of the above, from the allocator given at creation
};

namespace nvtext_amd {
namespace {

#include "codepoint_tables.inc"

constexpr uint32_t kCodepoints   = 0x110000;
constexpr uint32_t kDefaultEntry = 5u << 24;

// categories of an entry (cpp/src/text/detail/cp_data.h, read through the accessors of normalize.cu:44-98)
constexpr uint32_t kPad = 0, kPadIfLower = 1, kRemove = 2, kRemoveIfLower = 3, kReplace = 4;

constexpr int kNormThreads = 256;
constexpr int kNormItems   = 8;     // consecutive input bytes per lane
constexpr int kNormTile    = kNormThreads * kNormItems;  // input bytes per workgroup
constexpr int kBefore      = 5;   // a '[' this many bytes before the tile can still change the tile's slots
constexpr int kAfter       = 6;   // a '[' of the tile reads slots this many bytes past it
constexpr int kSlotBase    = 8;   // index of the tile's first position in the slot arrays (>= kBefore; 8 keeps a lane's bytes aligned)
constexpr int kSlots       = kSlotBase + kNormTile + 8;
constexpr int kRawBefore   = 8;   // bytes staged before the tile (>= kBefore)
constexpr int kRawAfter    = 12;  // bytes staged after it (>= kAfter + 3 for the longest character)
constexpr int kRawWords    = (kNormTile + kRawBefore + kRawAfter + 15 + 15) / 16 * 4;  // whole 16-byte blocks, any alignment
constexpr int32_t kSmallRows     = 131072;  // a column of so many rows is worked on before its size is known (see nvtext_amd_normalize_characters)
constexpr int64_t kSmallRowBytes = 4096;
constexpr int64_t kSmallLeast    = 256 << 10;
constexpr int64_t kSmallBytes    = 20 << 20;  // (40 MB of mixed text that way 130 us, as a large column 103; 18 MB 72 and 74)
constexpr int kStageBytes  = 4 * kNormTile;  // output bytes of a tile that are assembled in LDS; a tile with more writes them one by one

constexpr uint32_t kNotShort = 0x80000000u;  // beside the bytes of a string: there are more than eight, or it is the " [ " that may open a special token

struct NormTables {
  const uint32_t* ascii;  // 256 entries: the slots of the code points below 0x80, then zeros (a byte that is no such character gives nothing)
  const uint4* bmp;       // 65536 entries: the three slots and their bytes together, of the code points below 0x10000; and 65536
                          // more: those slots side by side, as a string of up to 12 bytes, and its bytes (with kNotShort)
  const uint8_t* sizes;   // 65536: the bytes alone (in a sixteenth of the memory, for the pass that counts)
  const uint32_t* entries;
  const uint64_t* second;
  const uint8_t* token_chars;
  const int32_t* token_offset;
  int32_t tokens;
  int32_t do_lower;
};

// cudf::strings::detail::codepoint_to_utf8 then from_char_utf8 (cpp/include/cudf/strings/detail/utf8.hpp:170-197,
// 143-168): the bytes of the character, first byte in the low bits, as the reference leaves them in a slot.
__host__ __device__ __forceinline__ uint32_t utf8_le(uint32_t cp)
{
  if (cp < 0x80u) return cp;
  uint32_t const t0 = 0x80u | (cp & 0x3Fu);
  uint32_t const t1 = 0x80u | ((cp >> 6) & 0x3Fu);
  if (cp < 0x800u) return (0xC0u | (cp >> 6)) | (t0 << 8);
  uint32_t const t2 = 0x80u | ((cp >> 12) & 0x3Fu);
  if (cp < 0x10000u) return (0xE0u | (cp >> 12)) | (t1 << 8) | (t0 << 16);
  return (0xF0u | ((cp >> 18) & 0x07u)) | (t2 << 8) | (t1 << 16) | (t0 << 24);
}

__host__ __device__ __forceinline__ uint32_t bytes_of(uint32_t slot)
{
#ifdef __HIP_DEVICE_COMPILE__
  return (39u - static_cast<uint32_t>(__clz(slot))) >> 3;
#else
  return (slot != 0) + (slot > 0xFFu) + (slot > 0xFFFFu) + (slot > 0xFFFFFFu);
#endif
}

// The code point of the character that starts with b0, the next bytes being b1..b3
// (to_char_utf8 and utf8_to_codepoint, cpp/include/cudf/strings/detail/utf8.hpp:68-97,118-140: the first byte
// alone says how many bytes belong to the character).
__device__ __forceinline__ uint32_t decode(uint32_t b0, uint32_t b1, uint32_t b2, uint32_t b3)
{
  if (b0 < 0x80u) return b0;
  if (b0 < 0xE0u) return ((b0 & 0x1Fu) << 6) | (b1 & 0x3Fu);
  if (b0 < 0xF0u) return ((b0 & 0x0Fu) << 12) | ((b1 & 0x3Fu) << 6) | (b2 & 0x3Fu);
  // packed value above 0xF8000000 decodes to 0
  uint32_t const packed = (b0 << 24) | (b1 << 16) | (b2 << 8) | b3;
  if (packed > 0xF8000000u) return 0u;
  return ((b0 & 0x07u) << 18) | ((b1 & 0x3Fu) << 12) | ((b2 & 0x3Fu) << 6) | (b3 & 0x3Fu);
}

// The slots of one code point (data_normalizer_kernel, cpp/src/text/normalize.cu:331-378).
__host__ __device__ __forceinline__ void slots_of(uint32_t cp, NormTables const& t, uint32_t& s0, uint32_t& s1, uint32_t& s2)
{
  s0 = s1 = s2       = 0;
  uint32_t const e   = cp < kCodepoints ? t.entries[cp] : kDefaultEntry;
  uint32_t const cat = (e >> 24) & 7u;
  bool const lower   = t.do_lower != 0;
  if (cat == kRemove || (lower && cat == kRemoveIfLower)) return;
  uint32_t const repl = (lower || cat == kReplace) ? (e & 0x1FFFFFu) : cp;
  uint32_t const r0   = repl ? repl : cp;
  if (lower && ((e >> 23) & 1u)) {  // two or three code points, never padded
    uint64_t const next = t.second[cp];
    uint32_t const r1 = static_cast<uint32_t>(next >> 32), r2 = static_cast<uint32_t>(next);
    s0 = utf8_le(r0);
    s1 = r1 ? utf8_le(r1) : 0u;
    s2 = r2 ? utf8_le(r2) : 0u;
    return;
  }
  uint32_t const one = utf8_le(r0);
  if (cat == kPad || (lower && cat == kPadIfLower)) {
    s0 = s2 = 0x20u;
    s1      = one;
  } else {
    s0 = one;
  }
}

constexpr int kWaveLeads = 256;  // first bytes of longer characters per wavefront (512 input bytes) that the counting pass lists: two in four bytes

template <bool SLOTS>
struct NormLds {
  alignas(16) uint32_t raw[kRawWords];  // the input bytes of the tile and its surroundings, zero outside the column
  uint32_t ascii[256];                 // code points below 0x80: slot 0 | slot 1 << 8 | slot 2 << 16 | bytes << 24; then zeros
  uint8_t sizes[SLOTS ? 4 : 256];      // their bytes (the pass that counts)
  union {
    // first byte of slot k of tile position i - kSlotBase; only filled where special tokens can be.  A first byte
    // tells '[', ']', a space and a-z from everything else, which is all the special tokens look at or change.
    alignas(8) uint8_t slot[3][kSlots];
    uint32_t staged[(kStageBytes + 8) / 4 + 4];  // afterwards: the tile's output bytes (and room for the dwords of a string that starts at the last one)
  };
  union {
    alignas(16) uint16_t prefix[kNormTile + 8];  // bytes the tile writes before each position; [tile] = all of them
    uint16_t lead_pos[kNormThreads / kWave][kWaveLeads];  // (before that: where in raw the longer characters of a wavefront begin)
  };
  uint32_t scan[kNormThreads / kWave + 1];
  uint32_t bracket;  // some lane of the tile saw what can open a special token
};

// The slots of the tile positions a lane owns (kNormItems * lane ..): consecutive bytes in, consecutive bytes out.
struct Owned {
  uint32_t s[kNormItems][3];
  uint32_t widest;  // the most bytes of a position, or somewhat more (the pass that writes)
};

// Slot `at` of the flat slot sequence (three per position).
template <bool S>
__device__ __forceinline__ uint8_t& flat_slot(NormLds<S>& lds, int at) { return lds.slot[at % 3][at / 3]; }

__device__ __forceinline__ bool has_byte(uint32_t v, uint32_t byte)
{
  uint32_t const x = v ^ (byte * 0x01010101u);
  return ((x - 0x01010101u) & ~x & 0x80808080u) != 0u;
}

// Bit 7 of every byte of v that is `byte`.
__device__ __forceinline__ uint64_t bytes_equal(uint64_t v, uint32_t byte)
{
  uint64_t const low = 0x7F7F7F7F7F7F7F7Full, x = v ^ (byte * 0x0101010101010101ull);
  return ~(((x & low) + low) | x | low);
}

// What may be a special token: its characters, spaces and empty slots left out, eight to a word and the first on top.
constexpr int kCandidateWords = 3;
struct Candidate {
  uint64_t word[kCandidateWords];
  int32_t size;  // 18 at most
};

// < 0, 0, > 0 as the candidate sorts before, equal to or after special token `i`.  (Behind their ends both are zeros: where
// those decide, the shorter one is the smaller.)
__device__ __forceinline__ int compare_candidate(Candidate const& c, NormTables const& t, int32_t i)
{
  int32_t const at = t.token_offset[i], size = t.token_offset[i + 1] - at;
#pragma unroll
  for (int w = 0; w < kCandidateWords; ++w) {
    uint64_t token = 0;
    if (8 * w < size) {
      __builtin_memcpy(&token, t.token_chars + at + 8 * w, 8);  // (there are eight bytes more than the tokens')
      token = __builtin_bswap64(token);
      if (size - 8 * w < 8) token &= ~0ull << (8 * (8 * w + 8 - size));
    }
    if (c.word[w] != token) return c.word[w] < token ? -1 : 1;
  }
  return c.size < size ? -1 : c.size > size ? 1 : 0;
}

// Whether a special token opens at slot index i (its slot 1 holds '['): the flat slot of its ']' if so, else -1.
// special_tokens_kernel, cpp/src/text/normalize.cu:283-301.  The 21 slots of seven positions are read at once and searched
// in registers: one by one from LDS, with a token's bytes one by one from memory, most of the time of text with tokens was
// that of the reads (200 MB with a token every 280 bytes 3778 -> 2747 us, every 2800 bytes 2039 -> 1706).
template <bool S>
__device__ int token_opens_at(NormLds<S>& lds, NormTables const& t, int i)
{
  if (lds.slot[1][i] != '[') return -1;
  uint64_t slot[3], closing[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    __builtin_memcpy(&slot[k], &lds.slot[k][i], 8);
    closing[k] = bytes_equal(slot[k], ']');
  }
  // the first ']' of the 17 slots after the '[' and the one behind it: slot k of position p is number 3 * p + k, numbers 2..18
  closing[0] &= 0x00FFFFFFFFFFFF00ull;
  closing[1] &= 0x0000FFFFFFFFFF00ull;
  closing[2] &= 0x0000FFFFFFFFFFFFull;
  int last = 99;
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (closing[k] != 0) last = min(last, 3 * (__builtin_ctzll(closing[k]) >> 3) + k);
  if (last == 99) return -1;
  Candidate c{};
  uint64_t word = 0;
  for (int at = 1, k = 1; at <= last; ++at) {
    uint32_t const b = static_cast<uint32_t>(k == 0 ? slot[0] : k == 1 ? slot[1] : slot[2]) & 0xFFu;
    if (b != 0u && b != 0x20u) {
      word = (word << 8) | b;
      ++c.size;
      if (c.size == 8) {
        c.word[0] = word;
        word      = 0;
      } else if (c.size == 16) {
        c.word[1] = word;
        word      = 0;
      }
    }
    if (++k == 3) {
      k = 0;
      slot[0] >>= 8;
      slot[1] >>= 8;
      slot[2] >>= 8;
    }
  }
  if ((c.size & 7) != 0) {
    word <<= 8 * (8 - (c.size & 7));
    if (c.size < 8) c.word[0] = word;
    else if (c.size < 16) c.word[1] = word;
    else c.word[2] = word;
  }
  int32_t first = 0, count = t.tokens;  // thrust::binary_search: lower_bound by halving, then !(value < *it)
  while (count > 0) {
    int32_t const half = count >> 1;
    if (compare_candidate(c, t, first + half) > 0) {
      first += half + 1;
      count -= half + 1;
    } else {
      count = half;
    }
  }
  if (first >= t.tokens || compare_candidate(c, t, first) < 0) return -1;
  return 3 * i + last;
}

// special_tokens_kernel (normalize.cu:270-316) over lds.slot, in two steps so that every decision reads unchanged
// slots.  A lane looks at its own positions; the first kBefore lanes also at the positions before the tile (a '['
// in the positions after the tile belongs to the next tile).
template <bool S>
__device__ void apply_special_tokens(NormLds<S>& lds, NormTables const& t, int tid)
{
  int found_to[kNormItems + 1];
#pragma unroll
  for (int k = 0; k <= kNormItems; ++k) {
    int const i = k < kNormItems ? kSlotBase + kNormItems * tid + k : kSlotBase - kBefore + tid;
    found_to[k] = (k < kNormItems || tid < kBefore) ? token_opens_at(lds, t, i) : -1;
  }
  lds_barrier();
#pragma unroll
  for (int k = 0; k <= kNormItems; ++k) {
    if (found_to[k] < 0) continue;
    int const i    = k < kNormItems ? kSlotBase + kNormItems * tid + k : kSlotBase - kBefore + tid;
    int const from = 3 * i + 1;
    flat_slot(lds, from + 1)        = 0u;  // the space after '['
    flat_slot(lds, found_to[k] - 1) = 0u;  // the space before ']'
    if (t.do_lower) {
      for (int at = from + 2; at < found_to[k] - 2; ++at) {
        uint32_t const c = flat_slot(lds, at);
        if (c >= 'a' && c <= 'z') flat_slot(lds, at) = static_cast<uint8_t>(c - 'a' + 'A');
      }
    }
  }
  lds_barrier();
}

// Code point of a character of two or three bytes whose bytes start `w` (first byte between 0xC0 and 0xEF): decode()
// without its branches.  The three bytes are turned round, a character of two bytes is moved to the end (0xC0..0xDF, which
// have bit 5 clear, look like a continuation byte there), and shifts to the right and masks, which take half the time of
// shifts to the left, put the pieces together: 21 cycles a wavefront instead of 40.
__device__ __forceinline__ uint32_t decode_short(uint32_t w)
{
  uint32_t const p = __builtin_amdgcn_perm(0u, w, 0x0c000102u) >> ((~w & 0x20u) >> 2);
  return ((p >> 4) & 0xF000u) | ((p >> 2) & 0x0FC0u) | (p & 0x3Fu);
}

// Slots of the character whose bytes start `w` (first byte in the low bits) and the bytes they hold together.  The
// Basic Multilingual Plane has them ready in one 16-byte table entry; the rest goes through the code point tables.
__device__ __forceinline__ uint32_t wide_slots(uint32_t w, NormTables const& t, uint32_t& s0, uint32_t& s1, uint32_t& s2)
{
  uint32_t cp = decode_short(w);
  if ((w & 0xFFu) >= 0xF0u) {  // four bytes (seldom)
    cp = decode(w & 0xFFu, (w >> 8) & 0xFFu, (w >> 16) & 0xFFu, w >> 24);
    if (cp >= 0x10000u) {
      slots_of(cp, t, s0, s1, s2);
      return bytes_of(s0) + bytes_of(s1) + bytes_of(s2);
    }
  }
  uint4 const e = t.bmp[cp];
  s0            = e.x;
  s1            = e.y;
  s2            = e.z;
  return e.w;
}

// The bytes of up to three slots side by side, first slot first: (lo, hi) = bytes 0..7 and 8..11.
__host__ __device__ __forceinline__ void slots_to_string(uint32_t s0, uint32_t s1, uint32_t s2, uint32_t& d0, uint32_t& d1, uint32_t& d2)
{
  uint32_t const b0  = bytes_of(s0);
  uint32_t const b01 = b0 + bytes_of(s1);  // <= 8
  uint64_t lo        = s0 | (static_cast<uint64_t>(s1) << (8u * b0));
  uint64_t const t   = s2;
  uint32_t const sh  = 8u * b01;
  lo |= b01 < 8u ? t << (sh & 63u) : 0ull;
  d2 = b01 >= 8u ? s2 : b01 > 4u ? static_cast<uint32_t>(t >> ((64u - sh) & 63u)) : 0u;
  d0 = static_cast<uint32_t>(lo);
  d1 = static_cast<uint32_t>(lo >> 32);
}

// The string that the character whose bytes start `w` turns into (12 bytes, zero padded), and its bytes.
__device__ __forceinline__ uint32_t wide_string(uint32_t w, NormTables const& t, uint32_t& d0, uint32_t& d1, uint32_t& d2)
{
  uint32_t cp = decode_short(w);
  if ((w & 0xFFu) >= 0xF0u) {
    cp = decode(w & 0xFFu, (w >> 8) & 0xFFu, (w >> 16) & 0xFFu, w >> 24);
    if (cp >= 0x10000u) {
      uint32_t s0, s1, s2;
      slots_of(cp, t, s0, s1, s2);
      slots_to_string(s0, s1, s2, d0, d1, d2);
      return bytes_of(s0) + bytes_of(s1) + bytes_of(s2);
    }
  }
  uint4 const e = t.bmp[0x10000u + cp];
  d0            = e.x;
  d1            = e.y;
  d2            = e.z;
  return e.w & 0xFFu;
}

// Bytes that the character whose bytes start `w` produces, without its slots; opener: whether it is a '['.
__device__ __forceinline__ uint32_t wide_size(uint32_t w, NormTables const& t, bool& opener)
{
  uint32_t cp = decode_short(w);
  if ((w & 0xFFu) >= 0xF0u) {
    cp = decode(w & 0xFFu, (w >> 8) & 0xFFu, (w >> 16) & 0xFFu, w >> 24);
    if (cp >= 0x10000u) {
      uint32_t s0, s1, s2;
      slots_of(cp, t, s0, s1, s2);
      return bytes_of(s0) + bytes_of(s1) + bytes_of(s2);
    }
  }
  opener = opener || cp == '[';
  return t.sizes[cp];
}

// The slots (and sizes) of the eight positions whose bytes are lo64; hi64 = bytes 4..11.  Returns the bytes they produce.
template <bool S>
__device__ __forceinline__ uint32_t owned_slots(NormLds<S> const& lds, uint64_t lo64, uint64_t hi64, NormTables const& t, Owned& mine,
                                                uint32_t (&size)[kNormItems])
{
  uint32_t sum = 0;
  // one-byte characters through the table; continuation bytes give nothing
#pragma unroll
  for (int j = 0; j < kNormItems; ++j) {
    uint32_t const b = static_cast<uint32_t>(lo64 >> (8 * j)) & 0xFFu;
    uint32_t const d = lds.ascii[b];
    mine.s[j][0]     = d & 0xFFu;
    mine.s[j][1]     = (d >> 8) & 0xFFu;
    mine.s[j][2]     = (d >> 16) & 0xFFu;
    size[j]          = d >> 24;
    sum += size[j];
  }
  // each first byte of a longer character (seldom more than four in eight bytes) goes through the code point tables
  uint64_t leads = lo64 & (lo64 << 1) & 0x8080808080808080ull;  // bit 7 of the bytes >= 0xC0
  while (leads) {
    int const at = (__ffsll(static_cast<long long>(leads)) - 1) >> 3;
    leads &= leads - 1ull;
    uint32_t const w = static_cast<uint32_t>((at < 4 ? lo64 : hi64) >> (8 * (at & 3)));
    uint32_t s0, s1, s2;
    uint32_t const bytes = wide_slots(w, t, s0, s1, s2);
    sum += bytes;
    // (as bit masks: written as "if (j == at)", the eight cases become a tree of branches, which lanes with
    // different `at` walk one leaf after the other)
#pragma unroll
    for (int j = 0; j < kNormItems; ++j) {
      uint32_t const here = static_cast<uint32_t>((static_cast<int32_t>(j ^ at) - 1) >> 31);  // all ones where j == at
      mine.s[j][0] = (mine.s[j][0] & ~here) | (s0 & here);
      mine.s[j][1] = (mine.s[j][1] & ~here) | (s1 & here);
      mine.s[j][2] = (mine.s[j][2] & ~here) | (s2 & here);
      size[j]      = (size[j] & ~here) | (bytes & here);
    }
  }
  return sum;
}

// owned_slots for the pass that writes: what each position turns into as a string of bytes (mine.s[j][0..2] = bytes
// 0..11, zero padded) instead of slots, ready to be placed.
template <bool S>
__device__ __forceinline__ uint32_t owned_strings(NormLds<S> const& lds, uint64_t lo64, uint64_t hi64, NormTables const& t, Owned& mine,
                                                  uint32_t (&size)[kNormItems])
{
  uint32_t sum = 0;
#pragma unroll
  for (int j = 0; j < kNormItems; ++j) {
    uint32_t const b = static_cast<uint32_t>(lo64 >> (8 * j)) & 0xFFu;
    uint32_t const d = lds.ascii[b];
    mine.s[j][0]     = d & 0xFFFFFFu;  // one byte per slot, empty slots last: the slots side by side are the string
    mine.s[j][1]     = 0u;
    mine.s[j][2]     = 0u;
    size[j]          = d >> 24;
    sum += size[j];
  }
  mine.widest    = 3u;
  uint64_t leads = lo64 & (lo64 << 1) & 0x8080808080808080ull;  // bit 7 of the bytes >= 0xC0
  while (leads) {
    int const at = (__ffsll(static_cast<long long>(leads)) - 1) >> 3;
    leads &= leads - 1ull;
    uint32_t const w = static_cast<uint32_t>((at < 4 ? lo64 : hi64) >> (8 * (at & 3)));
    uint32_t d0, d1, d2;
    uint32_t const bytes = wide_string(w, t, d0, d1, d2);
    sum += bytes;
    mine.widest = max(mine.widest, bytes);
#pragma unroll
    for (int j = 0; j < kNormItems; ++j) {
      uint32_t const here = static_cast<uint32_t>((static_cast<int32_t>(j ^ at) - 1) >> 31);  // all ones where j == at
      mine.s[j][0] = (mine.s[j][0] & ~here) | (d0 & here);
      mine.s[j][1] = (mine.s[j][1] & ~here) | (d1 & here);
      size[j]      = (size[j] & ~here) | (bytes & here);
    }
    if (ballot64(bytes > 8u) != 0) {  // (seldom: the third dwords are zeros otherwise)
#pragma unroll
      for (int j = 0; j < kNormItems; ++j) mine.s[j][2] = j == at ? d2 : mine.s[j][2];
    }
  }
  return sum;
}

__device__ __forceinline__ void wave_lds_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The bytes that the wavefront's 512 positions produce, for the pass that only sizes the output (a lane's return value
// holds the sizes of characters that are not its own: only the sum over the wavefront means something; so does `opener`,
// whether one of the longer characters is an over-long '[').
// One-byte characters go through the table in LDS, lanes <-> bytes.  The first bytes of longer characters are few
// and unevenly spread (none in English text, every other byte in Cyrillic or Greek), and each needs a read of a table
// by code point: the wavefront lists them and goes through the list lanes <-> characters, every lane at work.  Text
// has no more than two of them in four bytes, which is what the list is built for.
// `byte0` = the byte offset in lds.raw of the tile's first byte.
template <bool SLOTS>
__device__ __forceinline__ uint32_t owned_dense(NormLds<SLOTS>& lds, uint32_t own0, uint32_t own1, uint32_t next, uint32_t byte0, NormTables const& t,
                                                int tid, bool& opener)
{
  uint32_t sum = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) sum += lds.sizes[(own0 >> (8 * j)) & 0xFFu];
#pragma unroll
  for (int j = 0; j < 4; ++j) sum += lds.sizes[(own1 >> (8 * j)) & 0xFFu];
  uint32_t const leads0 = own0 & (own0 << 1) & 0x80808080u, leads1 = own1 & (own1 << 1) & 0x80808080u;  // bit 7 of the bytes >= 0xC0
  if (ballot64((leads0 | leads1) != 0u) == 0) return sum;
  uint32_t const more0 = leads0 & (leads0 - 1u), more1 = leads1 & (leads1 - 1u);
  if (ballot64(((more0 & (more0 - 1u)) | (more1 & (more1 - 1u))) != 0u) != 0) {
    // three of four bytes begin a character: not text; every lane walks its own
    uint64_t const lo64 = (static_cast<uint64_t>(own1) << 32) | own0, hi64 = (static_cast<uint64_t>(next) << 32) | own1;
    uint64_t l          = (static_cast<uint64_t>(leads1) << 32) | leads0;
    while (l) {
      int const at = (__ffsll(static_cast<long long>(l)) - 1) >> 3;
      l &= l - 1ull;
      sum += wide_size(static_cast<uint32_t>((at < 4 ? lo64 : hi64) >> (8 * (at & 3))), t, opener);
    }
    return sum;
  }
  uint32_t const n0   = static_cast<uint32_t>(__builtin_popcount(leads0));
  uint32_t const n    = n0 + static_cast<uint32_t>(__builtin_popcount(leads1));
  uint32_t const incl = wave_inclusive_scan(n);
  uint32_t const all  = wave_bcast(incl, kWave - 1);
  uint16_t* const list = lds.lead_pos[tid / kWave];
  {
    uint32_t const at = byte0 + kNormItems * tid;
    uint16_t* to      = list + (incl - n);
    if (leads0 != 0u) to[0] = static_cast<uint16_t>(at + (static_cast<uint32_t>(__builtin_ctz(leads0)) >> 3));
    if (more0 != 0u) to[1] = static_cast<uint16_t>(at + (static_cast<uint32_t>(__builtin_ctz(more0)) >> 3));
    to += n0;
    if (leads1 != 0u) to[0] = static_cast<uint16_t>(at + 4u + (static_cast<uint32_t>(__builtin_ctz(leads1)) >> 3));
    if (more1 != 0u) to[1] = static_cast<uint16_t>(at + 4u + (static_cast<uint32_t>(__builtin_ctz(more1)) >> 3));
  }
  wave_lds_sync();
  for (uint32_t r = lane_id(); r < all; r += kWave) {
    uint32_t const off = list[r];
    uint32_t const w   = __builtin_amdgcn_alignbit(lds.raw[(off >> 2) + 1], lds.raw[off >> 2], 8u * (off & 3u));
    sum += wide_size(w, t, opener);
  }
  return sum;
}

// v, of which the compiler does not know that it is the same in every trip of a loop: it keeps no sums of it over the trips
// then, for which it would spill registers (normalize_count_small_kernel: 128 and 74 spilled -> 91 and none; 20000 rows of
// 300 bytes 70 -> 35 us a call).
__device__ __forceinline__ int same_again(int v)
{
  asm volatile("" : "+v"(v));
  return v;
}

// The 16 bytes at `block`, which are the column's bytes from position p on; bytes outside [0, n) read as 0.
__device__ __forceinline__ uint4 load_within(const uint4* block, int64_t p, int64_t n)
{
  uint4 v = make_uint4(0u, 0u, 0u, 0u);
  if (p + 15 >= 0 && p < n) {
    v = load_stream(block);
    if (p < 0 || p + 16 > n) {  // the first or the last block of the column: clear what lies outside
      uint32_t* const part = &v.x;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        int64_t const q = p + 4 * k;
        uint32_t keep   = 0xFFFFFFFFu;
        if (q < 0) keep = q <= -4 ? 0u : keep << (8 * static_cast<uint32_t>(-q));
        if (q + 4 > n) keep = q >= n ? 0u : keep & (0xFFFFFFFFu >> (8 * static_cast<uint32_t>(q + 4 - n)));
        part[k] &= keep;
      }
    }
  }
  return v;
}

// Whether everything that is staged of the tile at t0 lies within the column.
__device__ __forceinline__ bool tile_is_inside(int64_t t0, int64_t n) { return t0 >= kRawBefore + 15 && t0 + 4 * kRawWords - kRawBefore <= n; }

// The lane's eight bytes of a tile and the four after them, the tile staged in LDS with its surroundings, the ASCII table
// beside it; `mis`: what the tile's alignment puts in front of them.
struct OwnBytes {
  uint32_t own0, own1, next;
  uint32_t mis;
};
template <bool SLOTS>
__device__ __forceinline__ OwnBytes stage_tile(NormLds<SLOTS>& lds, const uint8_t* chars, int64_t t0, int64_t n, NormTables const& t, int tid)
{
  // stage [t0 - kRawBefore, t0 + kNormTile + kRawAfter) with one aligned 16-byte load per lane (the first 131 lanes);
  // bytes outside [0, n) read as 0.  Everything is requested before anything is waited for.
  static_assert(kNormThreads == 256, "a table entry per lane");
  uint32_t const table_entry = t.ascii[tid];
  const uint8_t* const wb    = chars + t0 - kRawBefore;
  uint32_t const mis         = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(wb) & 15u);
  if (tid < kRawWords / 4) {
    int64_t const p = t0 - kRawBefore - mis + 16 * static_cast<int64_t>(tid);  // column position of the block's first byte
    const uint4* const block = reinterpret_cast<const uint4*>(wb - mis) + tid;
    uint4 const v            = tile_is_inside(t0, n) ? load_stream(block) : load_within(block, p, n);
    *reinterpret_cast<uint4*>(&lds.raw[4 * tid]) = v;
  }
  lds.ascii[tid] = table_entry;
  if constexpr (!SLOTS) lds.sizes[tid] = static_cast<uint8_t>(table_entry >> 24);
  if (tid == 0) lds.bracket = 0u;
  lds_barrier();

  // the lane's eight bytes and the four after them, whatever the alignment of the tile in memory
  uint32_t const shift = 8u * (mis & 3u);
  int const word       = static_cast<int>((mis + kRawBefore) >> 2) + 2 * tid;
  uint32_t const r0 = lds.raw[word], r1 = lds.raw[word + 1], r2 = lds.raw[word + 2], r3 = lds.raw[word + 3];
  uint32_t const own0 = __builtin_amdgcn_alignbit(r1, r0, shift);
  uint32_t const own1 = __builtin_amdgcn_alignbit(r2, r1, shift);
  uint32_t const next = __builtin_amdgcn_alignbit(r3, r2, shift);
  return OwnBytes{own0, own1, next, mis};
}

// Whether a special token may open in one of the eight positions before the tile (five needed): the first eight lanes
// decode the character that begins at theirs, so that an over-long '[' is one here exactly if it is one to the slots.
// Both passes ask this: one that took a tile for free of tokens while the other applied them would give it another size.
__device__ __forceinline__ bool opener_before(const uint32_t* raw, uint32_t lane, uint32_t mis)
{
  if (lane >= kRawBefore) return false;
  uint32_t const off = mis + lane;
  uint32_t const w   = __builtin_amdgcn_alignbit(raw[(off >> 2) + 1], raw[off >> 2], 8u * (off & 3u));
  uint32_t const b0  = w & 0xFFu;
  return b0 < 0xC0u ? b0 == '[' : decode(b0, (w >> 8) & 0xFFu, (w >> 16) & 0xFFu, w >> 24) == '[';
}

// One tile: the slots of the lane's positions, special tokens applied.  Returns the bytes they produce.  Without
// SLOTS only that number is wanted: the slots are then built only in tiles that may hold a special token.  MARKED: the tile
// is known to be one.
template <bool SLOTS, bool MARKED = false>
__device__ __forceinline__ uint32_t tile_slots(NormLds<SLOTS>& lds, const uint8_t* chars, int64_t t0, int64_t n, NormTables const& t, int tid,
                                               Owned& mine, uint32_t (&size)[kNormItems])
{
  OwnBytes const own = stage_tile(lds, chars, t0, n, t, tid);
  uint32_t const own0 = own.own0, own1 = own.own1, next = own.next, mis = own.mis;
  uint64_t const lo64 = (static_cast<uint64_t>(own1) << 32) | own0;
  uint64_t const hi64 = (static_cast<uint64_t>(next) << 32) | own1;
  // (the pass that wants the slots keeps them in registers all the way: listing the longer characters for it as well
  // saves it 4 % of its instructions and costs it two of its seven wavefronts per SIMD, 8.6 -> 10.7 ms on the
  // multilingual workload; the pass that only counts gains 13 % from the list)
  uint32_t sum  = 0;
  bool overlong = false;
  if constexpr (SLOTS) sum = owned_strings(lds, lo64, hi64, t, mine, size);
  else if constexpr (!MARKED) sum = owned_dense(lds, own0, own1, next, mis + kRawBefore, t, tid, overlong);

  if (t.tokens > 0) {
    // A special token starts at a position whose slot 1 is '['.  Tiles without one skip the exchange through LDS.
    // No code point's replacement is a '[', so it takes a '[' byte or an over-long encoding of it: that is what
    // decides when the slots have not been built.
    if constexpr (!MARKED) {
      bool bracket = opener_before(lds.raw, tid, mis);
      if constexpr (SLOTS) {
        // (strings: a '[' is padded like all punctuation, so it is the middle byte of " [ ")
#pragma unroll
        for (int j = 0; j < kNormItems; ++j) bracket |= ((mine.s[j][0] >> 8) & 0xFFu) == '[';
      } else {
        bracket = bracket || overlong || has_byte(own0, '[') || has_byte(own1, '[');
      }
      if (ballot64(bracket) != 0 && lane_id() == 0) lds.bracket = 1u;
      lds_barrier();
    }
    if (MARKED || lds.bracket != 0u) {
      owned_slots(lds, lo64, hi64, t, mine, size);  // (the slots themselves, whatever mine held)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        uint32_t a = 0, b = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          a |= (mine.s[j][k] & 0xFFu) << (8 * j);
          b |= (mine.s[j + 4][k] & 0xFFu) << (8 * j);
        }
        *reinterpret_cast<uint2*>(&lds.slot[k][kSlotBase + kNormItems * tid]) = make_uint2(a, b);
      }
      if (tid < kBefore + kAfter) {  // the positions either side of the tile
        int const pos             = tid < kBefore ? tid - kBefore : kNormTile + tid - kBefore;
        const uint8_t* const rawb = reinterpret_cast<const uint8_t*>(lds.raw) + mis + kRawBefore + pos;
        uint32_t const b0         = rawb[0];
        uint32_t s0 = 0, s1 = 0, s2 = 0;
        if (b0 < 0x80u) {
          uint32_t const d = lds.ascii[b0];
          s0               = d & 0xFFu;
          s1               = (d >> 8) & 0xFFu;
          s2               = (d >> 16) & 0xFFu;
        } else if (b0 >= 0xC0u) {
          wide_slots(b0 | (static_cast<uint32_t>(rawb[1]) << 8) | (static_cast<uint32_t>(rawb[2]) << 16) | (static_cast<uint32_t>(rawb[3]) << 24),
                     t, s0, s1, s2);
        }
        lds.slot[0][kSlotBase + pos] = static_cast<uint8_t>(s0);
        lds.slot[1][kSlotBase + pos] = static_cast<uint8_t>(s1);
        lds.slot[2][kSlotBase + pos] = static_cast<uint8_t>(s2);
      }
      lds_barrier();
      apply_special_tokens(lds, t, tid);
      // the tokens only ever empty a slot or turn its letter into upper case: take over the first bytes that changed
      sum         = 0;
      mine.widest = 0;
#pragma unroll
      for (int j = 0; j < kNormItems; ++j) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          uint32_t const now = lds.slot[k][kSlotBase + kNormItems * tid + j];
          if (now != (mine.s[j][k] & 0xFFu)) mine.s[j][k] = now;
        }
        // keep the filled slots of a position in front (the output is the same): the writer relies on it
#pragma unroll
        for (int again = 0; again < 2; ++again) {
          if (mine.s[j][0] == 0u) {
            mine.s[j][0] = mine.s[j][1];
            mine.s[j][1] = mine.s[j][2];
            mine.s[j][2] = 0u;
          }
        }
        if (mine.s[j][1] == 0u) {
          mine.s[j][1] = mine.s[j][2];
          mine.s[j][2] = 0u;
        }
        size[j] = bytes_of(mine.s[j][0]) + bytes_of(mine.s[j][1]) + bytes_of(mine.s[j][2]);
        sum += size[j];
        mine.widest = max(mine.widest, size[j]);
        if (SLOTS) slots_to_string(mine.s[j][0], mine.s[j][1], mine.s[j][2], mine.s[j][0], mine.s[j][1], mine.s[j][2]);
      }
    }
  }
  return sum;
}

// tile_bytes[tile] = bytes the tile's input positions produce
__global__ void __launch_bounds__(kNormThreads, 8) normalize_count_kernel(const uint8_t* __restrict__ chars, int64_t n, NormTables t,
                                                                       uint32_t* __restrict__ tile_bytes)
{
  __shared__ NormLds<false> lds;
  int const tid    = threadIdx.x;
  int64_t const t0 = static_cast<int64_t>(blockIdx.x) * kNormTile;
  Owned mine;
  uint32_t size[kNormItems];
  uint32_t const sum = tile_slots<false>(lds, chars, t0, n, t, tid, mine, size);
  uint32_t total;
  block_exclusive_scan_lds<kNormThreads>(sum, lds.scan, &total);
  if (threadIdx.x == 0) tile_bytes[blockIdx.x] = total;
}

// The same for a column of many tiles: every wavefront takes a whole one, with a list of its longer characters, and waits
// for no other.  Tiles that may hold a special token are left for the workgroup to do together at the end, as
// normalize_count_kernel does them.
// What bounds it is instructions again: with a workgroup a tile half the time went on barriers, on starting, on staging
// the table and on a list for every 512 bytes.  766 MB of mixed text 461 -> 255 to 266 us (traced); several tiles for a wavefront, with the bytes
// of the next one on their way, no faster.  A small column has too few wavefronts this way: with both passes by workgroups below 12,288
// tiles, or by wavefronts from 4,096 on, 8.5 MB of mixed text take 43.9 and 46.9 us, 18 MB 75.6 and 71, of ASCII 40.9 and 38.8, 65 and 57.
constexpr int kTileWaves          = kNormThreads / kWave;
constexpr int kLaneWords          = kNormTile / kWave / 4;  // dwords of a tile per lane, two of every 512 bytes
constexpr int64_t kManyTiles      = 8192;                   // a column of so many tiles
// Whether there is nothing for the end.  (Asked before the loop over the four: what the compiler gets ready for that loop it spills
// to memory, 5 GB of HBM writes beside the 4.2 GB of a result.)
__device__ __forceinline__ bool none_left(const uint32_t (&left)[kTileWaves])
{
  uint32_t any = 0;
#pragma unroll
  for (int k = 0; k < kTileWaves; ++k) any |= left[k];
  return __builtin_amdgcn_readfirstlane(static_cast<int>(any)) == 0;
}

union CountLds {
  struct {
    alignas(16) uint32_t raw[kTileWaves][kRawWords];
    uint16_t leads[kTileWaves][kNormTile / 2];  // where in raw the longer characters of a tile begin
  };
  NormLds<false> tile;
};
__global__ void __launch_bounds__(kNormThreads, 8) normalize_count_tiles_kernel(const uint8_t* __restrict__ chars, int64_t n, uint32_t tiles,
                                                                             NormTables t, uint32_t* __restrict__ tile_bytes)
{
  __shared__ CountLds lds;
  __shared__ uint8_t sizes[256];
  __shared__ uint32_t left[kTileWaves];  // the tiles left for the end
  uint32_t const wave  = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = lane_id();
  uint32_t const tile0 = blockIdx.x * kTileWaves, tile = tile0 + wave;
  int64_t const t0     = static_cast<int64_t>(tile) * kNormTile;
  uint32_t const mis   = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(chars - kRawBefore) & 15u);  // (of every tile: they are 2048 bytes apart)
  uint32_t* const raw  = lds.raw[wave];
  bool opener          = false;
  uint32_t const table_entry = t.ascii[threadIdx.x];
  bool const third = lane < kRawWords / 4 - 2 * kWave;
  uint4 v[3];
  if (tile < tiles) {
    const uint4* const block = reinterpret_cast<const uint4*>(chars + t0 - kRawBefore - mis) + lane;
    if (tile_is_inside(t0, n)) {
      v[0] = load_stream(block);
      v[1] = load_stream(block + kWave);
      if (third) v[2] = load_stream(block + 2 * kWave);
    } else {
      int64_t const p = t0 - kRawBefore - mis + 16 * static_cast<int64_t>(lane);
      v[0]            = load_within(block, p, n);
      v[1]            = load_within(block + kWave, p + 16 * kWave, n);
      if (third) v[2] = load_within(block + 2 * kWave, p + 32 * kWave, n);
    }
  }
  sizes[threadIdx.x] = static_cast<uint8_t>(table_entry >> 24);
  lds_barrier();
  bool marked = false;
  if (tile < tiles) {
    reinterpret_cast<uint4*>(raw)[lane]         = v[0];
    reinterpret_cast<uint4*>(raw)[lane + kWave] = v[1];
    if (third) reinterpret_cast<uint4*>(raw)[lane + 2 * kWave] = v[2];
    wave_lds_sync();
    const uint32_t* const own_raw = raw + ((mis + kRawBefore) >> 2) + 2 * lane;
    uint32_t const shift          = 8u * (mis & 3u);
    uint32_t sum = 0, many = 0, n_leads = 0;
    uint32_t leads[kLaneWords];  // bit 7 of the bytes >= 0xC0
#pragma unroll
    for (int q = 0; q < kLaneWords / 2; ++q) {
      const uint32_t* const r = own_raw + q * (2 * kWave);
      uint32_t const r0 = r[0], r1 = r[1], r2 = r[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t const own = h ? __builtin_amdgcn_alignbit(r2, r1, shift) : __builtin_amdgcn_alignbit(r1, r0, shift);
#pragma unroll
        for (int j = 0; j < 4; ++j) sum += sizes[(own >> (8 * j)) & 0xFFu];
        uint32_t const l    = own & (own << 1) & 0x80808080u;
        uint32_t const more = l & (l - 1u);
        leads[2 * q + h]    = l;
        many |= more & (more - 1u);
        n_leads += static_cast<uint32_t>(__builtin_popcount(l));
        opener = opener || has_byte(own, '[');
      }
    }
    opener = opener || opener_before(raw, lane, mis);
    marked = t.tokens > 0 && ballot64(opener) != 0;
    if (!marked && ballot64(n_leads != 0u) != 0) {
      uint32_t const at = mis + kRawBefore + kNormItems * lane;
      if (ballot64(many != 0u) != 0) {
        // three of four bytes begin a character: not text; every lane walks its own
#pragma unroll
        for (int k = 0; k < kLaneWords; ++k) {
          uint32_t l = leads[k];
          while (l != 0u) {
            uint32_t const off = at + (k / 2) * (kWave * kNormItems) + 4 * (k & 1) + (static_cast<uint32_t>(__builtin_ctz(l)) >> 3);
            l &= l - 1u;
            sum += wide_size(__builtin_amdgcn_alignbit(raw[(off >> 2) + 1], raw[off >> 2], 8u * (off & 3u)), t, opener);
          }
        }
      } else {
        uint32_t const incl  = wave_inclusive_scan(n_leads);
        uint32_t const all   = wave_bcast(incl, kWave - 1);
        uint16_t* const list = lds.leads[wave];
        uint16_t* to         = list + (incl - n_leads);
#pragma unroll
        for (int k = 0; k < kLaneWords; ++k) {
          uint32_t const l = leads[k], more = l & (l - 1u);
          uint32_t const off = at + (k / 2) * (kWave * kNormItems) + 4 * (k & 1);
          if (l != 0u) to[0] = static_cast<uint16_t>(off + (static_cast<uint32_t>(__builtin_ctz(l)) >> 3));
          if (more != 0u) to[1] = static_cast<uint16_t>(off + (static_cast<uint32_t>(__builtin_ctz(more)) >> 3));
          to += __builtin_popcount(l);
        }
        wave_lds_sync();
        for (uint32_t r = lane; r < all; r += kWave) {
          uint32_t const off = list[r];
          sum += wide_size(__builtin_amdgcn_alignbit(raw[(off >> 2) + 1], raw[off >> 2], 8u * (off & 3u)), t, opener);
        }
      }
    }
    marked = t.tokens > 0 && ballot64(opener) != 0;
    sum    = wave_inclusive_scan(sum);
    if (!marked && lane == kWave - 1) tile_bytes[tile] = sum;
  }
  if (t.tokens == 0) return;
  if (lane == 0) left[wave] = marked ? 1u : 0u;
  lds_barrier();
  if (none_left(left)) return;
#pragma unroll 1
  for (int k = 0; k < kTileWaves; ++k) {
    if (__builtin_amdgcn_readfirstlane(static_cast<int>(left[k])) == 0) continue;
    int const tid       = same_again(threadIdx.x);
    Owned mine;
    uint32_t size[kNormItems];
    uint32_t const bytes = tile_slots<false, true>(lds.tile, chars, static_cast<int64_t>(tile0 + k) * kNormTile, n, t, tid, mine, size);
    uint32_t total;
    block_exclusive_scan_lds<kNormThreads>(bytes, lds.tile.scan, &total);
    if (threadIdx.x == 0) tile_bytes[tile0 + k] = total;
    lds_barrier();
  }
}

// The same for a column whose size the host does not know yet: where its bytes lie the kernel reads from the offsets (a
// column of no bytes, or of more than most_bytes, is left alone), and a workgroup takes every gridDim.x-th tile.  The
// last wavefront also finds tile_row[tile], as normalize_tile_rows_kernel does, 64 rows looked at in one step.
__global__ void __launch_bounds__(kNormThreads, 4) normalize_count_small_kernel(ColView col, int64_t most_bytes, NormTables t,
                                                                             uint32_t* __restrict__ tile_bytes, int32_t* __restrict__ tile_row)
{
  __shared__ NormLds<false> lds;
  int64_t const first = col.off(0), n = col.off(col.size) - first;
  if (n <= 0 || n > most_bytes) return;
  int64_t const tiles = (n + kNormTile - 1) / kNormTile;
  for (int64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    int64_t const t0 = tile * kNormTile;
    if (threadIdx.x >= kNormThreads - kWave) {
      int64_t lo = 0, hi = static_cast<int64_t>(col.size) + 1;
      while (lo < hi) {
        int64_t const step   = (hi - lo + kWave - 1) / kWave;
        int64_t const at     = lo + step * lane_id();
        bool const before    = at < hi && col.off(at) - first < t0;
        int64_t const passed = __builtin_popcountll(ballot64(before));
        if (passed == 0) break;
        hi = min(hi, lo + passed * step);
        lo = lo + (passed - 1) * step + 1;
      }
      if (lane_id() == 0) tile_row[tile] = static_cast<int32_t>(lo);
    }
    int const tid = same_again(threadIdx.x);
    Owned mine;
    uint32_t size[kNormItems];
    uint32_t const sum = tile_slots<false>(lds, col.chars + first, t0, n, t, tid, mine, size);
    uint32_t total;
    block_exclusive_scan_lds<kNormThreads>(sum, lds.scan, &total);
    if (threadIdx.x == 0) tile_bytes[tile] = total;
    lds_barrier();
  }
}

// After that: the places of the tiles' bytes in the result (one workgroup), and what the host has to know: dst = {first
// byte, byte past the last, bytes of the result}.
constexpr int kFinishThreads = 1024;
__global__ void __launch_bounds__(kFinishThreads) normalize_finish_kernel(ColView col, int64_t most_bytes, const uint32_t* __restrict__ tile_bytes,
                                                                          uint64_t* __restrict__ tile_offset, uint64_t* __restrict__ dst, HostPost post)
{
  __shared__ uint64_t lds[kFinishThreads / kWave + 1];
  int64_t const first = col.off(0), last = col.off(col.size), n = last - first;
  int64_t const tiles = n > 0 && n <= most_bytes ? (n + kNormTile - 1) / kNormTile : 0;
  constexpr int kEach = 4;
  uint64_t carry      = 0;
  for (int64_t base = 0; base < tiles; base += kEach * kFinishThreads) {
    int64_t const i = base + kEach * static_cast<int64_t>(threadIdx.x);
    uint64_t v[kEach], sum = 0;
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
      v[k] = i + k < tiles ? tile_bytes[i + k] : 0;
      sum += v[k];
    }
    uint64_t total;
    uint64_t run = carry + block_exclusive_scan64<kFinishThreads>(sum, lds, &total);
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
      if (i + k < tiles) tile_offset[i + k] = run;
      run += v[k];
    }
    carry += total;
  }
  if (threadIdx.x == 0) {
    dst[0] = static_cast<uint64_t>(first);
    dst[1] = static_cast<uint64_t>(last);
    dst[2] = carry;
    post.send();
  }
}

// tile_row[tile] = the first row (of rows + 1: the end counts as one) whose first byte lies at or after the tile's
// first byte.  Eight lanes search for a tile in columns of up to kSearchTiles tiles, where it is the reads in a row that take the time (25 MB
// of mixed text 76.9 -> 74.4 us, 64 MB 133.2 -> 131.0, 200 MB 324 -> 323); beyond, where it is their number, a lane (600 MB 8.8 us,
// with eight 18.7).
constexpr int64_t kSearchTiles = 100'000;
template <int LANES>
__global__ void __launch_bounds__(256) normalize_tile_rows_kernel(ColView col, int64_t first, int64_t tiles, int32_t* __restrict__ tile_row)
{
  int64_t const tile    = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / LANES;
  uint32_t const member = threadIdx.x % LANES;
  int64_t const t0      = tile * kNormTile;
  uint32_t lo = 0, hi = tile < tiles ? static_cast<uint32_t>(col.size) + 1u : 0u;  // the answer lies in [lo, hi]
  if (LANES == 1) {
    while (lo < hi) {
      uint32_t const mid = lo + ((hi - lo) >> 1);
      if (col.off(mid) - first < t0) lo = mid + 1;
      else hi = mid;
    }
  } else {
    lo = search_by_lanes<LANES>(lo, hi, member, [&](uint32_t row) { return col.off(row) - first < t0; });
  }
  if (tile < tiles && member == 0) tile_row[tile] = static_cast<int32_t>(lo);
}

// The rows that start in a tile: looked up when the tile begins (the barriers do not wait for global loads, so that the
// lane's own is back when the tile is done), given their places at its end.
struct TileRows {
  int64_t my_row, row_end;
  uint32_t start_lo, start_hi;  // the raw offset entry of my_row; not touched before the end
  __device__ __forceinline__ void request(ColView const& col, const int32_t* tile_row, uint32_t tile, uint32_t tiles)
  {
    int64_t const rows = col.size;
    my_row             = static_cast<int64_t>(tile_row[tile]) + threadIdx.x;
    // the rows that start in this tile end where the next tile's begin (the last tile also takes the end of the last row)
    row_end  = tile + 1 == tiles ? rows + 1 : static_cast<int64_t>(tile_row[tile + 1]);
    start_lo = start_hi = 0;
    if (my_row <= rows) {
      if (col.is64) {
        uint2 const v = static_cast<const uint2*>(col.offsets)[my_row + col.offset];
        start_lo      = v.x;
        start_hi      = v.y;
      } else {
        start_lo = static_cast<const uint32_t*>(col.offsets)[my_row + col.offset];
      }
    }
  }
  // rows whose first byte lies in [t0, t1) -- in [t0, n] for the last tile -- start at base + prefix
  __device__ __forceinline__ void place(ColView const& col, int64_t first, int64_t t0, uint64_t base, const uint16_t* prefix, void* out_offsets,
                                        int offsets_are_int64) const
  {
    int64_t const my_start = (col.is64 ? static_cast<int64_t>((static_cast<uint64_t>(start_hi) << 32) | start_lo)
                                       : static_cast<int64_t>(static_cast<int32_t>(start_lo))) - first;
    for (int64_t r = my_row; r < row_end; r += kNormThreads) {  // (more than one trip only in a tile of very short rows)
      int64_t const p   = r == my_row ? my_start : col.off(r) - first;
      uint64_t const at = base + prefix[p - t0];
      if (offsets_are_int64) static_cast<int64_t*>(out_offsets)[r] = static_cast<int64_t>(at);
      else static_cast<int32_t*>(out_offsets)[r] = static_cast<int32_t>(at);
    }
  }
};

// The tile's bytes from LDS, where they lie as they will lie in memory from the dword at or below dst on, to memory.
__device__ __forceinline__ void store_staged(const uint32_t* staged, uint8_t* dst, uint32_t lead, uint32_t total)
{
  int const tid           = threadIdx.x;
  const uint8_t* const sb = reinterpret_cast<const uint8_t*>(staged);
  uint32_t const end      = lead + total;
  uint32_t const w_lo     = (lead + 3u) >> 2;
  uint32_t const w_hi     = end >> 2;
  uint32_t* const dw      = reinterpret_cast<uint32_t*>(dst - lead);
  for (uint32_t w = w_lo + tid; w < w_hi; w += kNormThreads) store_stream(dw + w, staged[w]);
  uint32_t const head_end   = min(4u * w_lo, end);
  uint32_t const tail_begin = max(4u * w_hi, head_end);
  if (tid < 4) {
    uint32_t const at = lead + tid;
    if (at < head_end) (dst - lead)[at] = sb[at];
  } else if (tid < 8) {
    uint32_t const at = tail_begin + (tid - 4);
    if (at < end) (dst - lead)[at] = sb[at];
  }
}

// The buffer that the output bytes are assembled in starts out as zeros.
__device__ __forceinline__ void clear_staged(NormLds<true>& lds)
{
  int const tid = threadIdx.x;
  for (int i = tid; i < static_cast<int>(sizeof(lds.staged) / 16); i += kNormThreads) reinterpret_cast<uint4*>(lds.staged)[i] = make_uint4(0u, 0u, 0u, 0u);
  if (tid < static_cast<int>(sizeof(lds.staged) % 16) / 4) lds.staged[sizeof(lds.staged) / 16 * 4 + tid] = 0u;
}

// A lane's eight one-byte characters (three bytes at most each, `text` in the low bytes, their number in the top one) in a
// wavefront that has no others: a position's bytes travel together, as one (unaligned) dword whose spare bytes the next
// positions overwrite.  A position that starts in the lane's last three bytes is skipped; those bytes are kept in `last`
// (the four bytes written last, newest on top) and stored one by one at the end.  o: where the lane's bytes go, sum: their
// number.
template <typename Text, typename Size>
__device__ __forceinline__ void place_short(uint8_t* sb, uint32_t o, uint32_t sum, Text const& text, Size const& size)
{
  uint32_t const mine_end = o + sum;
  uint32_t last           = 0;
#pragma unroll
  for (int j = 0; j < kNormItems; ++j) {
    uint32_t const three = text(j), n = size(j);
    if (n != 0u && o + 4u <= mine_end) __builtin_memcpy(sb + o, &three, 4);
    last = __builtin_amdgcn_alignbit(three, last, 8u * n);
    o += n;
  }
  if (sum >= 1u) sb[mine_end - 1u] = static_cast<uint8_t>(last >> 24);
  if (sum >= 2u) sb[mine_end - 2u] = static_cast<uint8_t>(last >> 16);
  if (sum >= 3u) sb[mine_end - 3u] = static_cast<uint8_t>(last >> 8);
}

// Writes the tile's bytes at tile_offset[tile] and the output offset of every row that starts in the tile.
__device__ __forceinline__ void write_tile(NormLds<true>& lds, uint32_t tile, uint32_t tiles, ColView const& col, int64_t first, int64_t n,
                                           NormTables const& t, const uint64_t* tile_offset, const int32_t* tile_row, uint8_t* out_chars,
                                           void* out_offsets, int offsets_are_int64, int tid)
{
  int64_t const t0     = static_cast<int64_t>(tile) * kNormTile;
  uint64_t const base  = tile_offset[tile];
  TileRows tile_rows;
  tile_rows.request(col, tile_row, tile, tiles);
  Owned mine;
  uint32_t size[kNormItems];
  uint32_t const sum = tile_slots<true>(lds, col.chars + first, t0, n, t, tid, mine, size);
  // the buffer that the output bytes are assembled in starts out as zeros (the scan's barriers stand between this
  // and the first byte placed); in a tile that went through the special tokens it lies where the slots' first bytes
  // were, which the other wavefronts may still be reading
  if (t.tokens > 0 && lds.bracket != 0u) lds_barrier();
  clear_staged(lds);
  uint32_t total;
  uint32_t const before = block_exclusive_scan_lds<kNormThreads>(sum, lds.scan, &total);
  {
    uint32_t run = before;
    uint32_t packed[kNormItems / 2];
#pragma unroll
    for (int j = 0; j < kNormItems; ++j) {
      if (j & 1) packed[j >> 1] |= run << 16;
      else packed[j >> 1] = run;
      run += size[j];
    }
    *reinterpret_cast<uint4*>(&lds.prefix[kNormItems * tid]) = make_uint4(packed[0], packed[1], packed[2], packed[3]);
    if (tid == kNormThreads - 1) lds.prefix[kNormTile] = static_cast<uint16_t>(run);
  }

  uint8_t* const dst = out_chars + base;
  if (total <= static_cast<uint32_t>(kStageBytes)) {
    // the output bytes, laid out in LDS as they will lie in memory relative to an aligned dword.  A slot is stored
    // as one (unaligned) dword wherever the three bytes that may follow it still belong to this lane: later slots
    // overwrite them.  The last slots of the lane go byte by byte.
    uint32_t const lead = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst) & 3u);
    uint8_t* const sb   = reinterpret_cast<uint8_t*>(lds.staged);
    uint32_t o          = lead + before;
    if (ballot64(mine.widest > 3u) == 0) {
      // no position of the wavefront turns into more than three bytes
      place_short(sb, o, sum, [&](int j) { return mine.s[j][0]; }, [&](int j) { return size[j]; });
    } else {
      // longer strings: every position's bytes (zero padded) are or-ed into the aligned dwords they fall into;
      // the buffer was cleared, and what the neighbours put into a shared dword is theirs
      bool const past8 = ballot64(mine.widest > 8u) != 0;
#pragma unroll
      for (int j = 0; j < kNormItems; ++j) {
        uint32_t const sh   = 8u * (o & 3u);
        uint32_t* const at  = lds.staged + (o >> 2);
        uint64_t const a    = static_cast<uint64_t>(mine.s[j][0]) << sh;
        uint64_t const b    = static_cast<uint64_t>(mine.s[j][1]) << sh;
        atomicOr(at, static_cast<uint32_t>(a));
        atomicOr(at + 1, static_cast<uint32_t>(a >> 32) | static_cast<uint32_t>(b));
        atomicOr(at + 2, static_cast<uint32_t>(b >> 32));
        if (past8) {  // (a character that turns into three characters of three bytes, or into characters beyond U+FFFF)
          uint64_t const c = static_cast<uint64_t>(mine.s[j][2]) << sh;
          atomicOr(at + 2, static_cast<uint32_t>(c));
          atomicOr(at + 3, static_cast<uint32_t>(c >> 32));
        }
        o += size[j];
      }
    }
    lds_barrier();
    store_staged(lds.staged, dst, lead, total);
  } else {
    // more than four output bytes per input byte (only input that is not UTF-8 gets there): byte by byte
    uint8_t* o = dst + before;
#pragma unroll
    for (int j = 0; j < kNormItems; ++j)
      for (uint32_t k = 0; k < size[j]; ++k) *o++ = static_cast<uint8_t>((k < 4 ? mine.s[j][0] : k < 8 ? mine.s[j][1] : mine.s[j][2]) >> (8u * (k & 3u)));
    lds_barrier();  // lds.prefix is complete for the rows below
  }

  tile_rows.place(col, first, t0, base, lds.prefix, out_offsets, offsets_are_int64);
}

// The same, done here for ordinary text; tiles that may hold a special token, characters that turn into more than eight
// bytes and more first bytes of longer characters side by side than text has go through write_tile().
// What bounds it is the number of vector instructions (400 a wavefront, issued in 83 % of the cycles).  A lane keeps its one-byte characters as the table gives them and
// up to four longer ones beside them, each in registers of its own (instead of a string for every position, into which
// a longer character was selected eight times); where each goes in the lane's output comes from the eight sizes, a byte
// each, multiplied by 0x01..01.
constexpr int kLongChars = 4;  // of two bytes and more in eight bytes
__global__ void __launch_bounds__(kNormThreads, 6) normalize_write_kernel(ColView col, int64_t first, int64_t n, NormTables t,
                                                                       const uint64_t* __restrict__ tile_offset,
                                                                       const int32_t* __restrict__ tile_row, uint8_t* __restrict__ out_chars,
                                                                       void* __restrict__ out_offsets, int offsets_are_int64)
{
  __shared__ NormLds<true> lds;
  int const tid       = threadIdx.x;
  uint32_t const tile = blockIdx.x;
  int64_t const t0    = static_cast<int64_t>(tile) * kNormTile;
  uint64_t const base = tile_offset[tile];
  TileRows tile_rows;
  tile_rows.request(col, tile_row, tile, gridDim.x);
  OwnBytes const own  = stage_tile(lds, col.chars + first, t0, n, t, tid);
  uint64_t const lo64 = (static_cast<uint64_t>(own.own1) << 32) | own.own0;
  uint64_t const hi64 = (static_cast<uint64_t>(own.next) << 32) | own.own1;
  uint32_t text[kNormItems];
#pragma unroll
  for (int j = 0; j < kNormItems; ++j) text[j] = lds.ascii[static_cast<uint32_t>(lo64 >> (8 * j)) & 0xFFu];
  // the sizes of the positions, a byte each
  auto const top_bytes = [](uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_amdgcn_perm(b, a, 0x0c0c0703u) | __builtin_amdgcn_perm(d, c, 0x07030c0cu);
  };
  uint64_t sizes = (static_cast<uint64_t>(top_bytes(text[4], text[5], text[6], text[7])) << 32) | top_bytes(text[0], text[1], text[2], text[3]);
  uint64_t leads = lo64 & (lo64 << 1) & 0x8080808080808080ull;  // bit 7 of the bytes >= 0xC0
  bool const any_long = ballot64(leads != 0) != 0;
  bool other          = false;  // the tile is not for this kernel
  uint32_t d0[kLongChars] = {}, d1[kLongChars] = {}, at8[kLongChars] = {};
  uint64_t holders[kLongChars] = {};  // the lanes that have a k-th longer character, whatever it turns into
  if (any_long) {
    // all reads of the table in flight together
    uint4 e[kLongChars];
#pragma unroll
    for (int k = 0; k < kLongChars; ++k) {
      bool const have    = leads != 0;
      holders[k]         = ballot64(have);
      uint32_t const bit = static_cast<uint32_t>(__builtin_ctzll(leads | 0x8000000000000000ull));  // 8 * position + 7
      leads &= leads - 1ull;
      at8[k]           = bit - 7u;
      uint32_t const w = static_cast<uint32_t>((bit < 32u ? lo64 : hi64) >> (at8[k] & 31u));
      e[k]             = make_uint4(0u, 0u, 0u, 0u);
      if (have) e[k] = t.bmp[0x10000u + decode_short(w)];
      if (ballot64(have && (w & 0xFFu) >= 0xF0u) != 0) {  // four bytes (seldom)
        if (have && (w & 0xFFu) >= 0xF0u) e[k].w = wide_string(w, t, e[k].x, e[k].y, e[k].z);
      }
    }
#pragma unroll
    for (int k = 0; k < kLongChars; ++k) {
      d0[k] = e[k].x;
      d1[k] = e[k].y;
      sizes += static_cast<uint64_t>(e[k].w) << at8[k];
      other = other || e[k].w > 8u || d0[k] == 0x205B20u;  // (" [ ": an over-long '[')
    }
  }
  other = other || leads != 0;
  if (t.tokens > 0) other = other || has_byte(own.own0, '[') || has_byte(own.own1, '[') || opener_before(lds.raw, tid, own.mis);
  if (ballot64(other) != 0 && lane_id() == 0) lds.bracket = 1u;
  clear_staged(lds);
  // where each position's bytes begin in the lane's: the sums of the sizes before it (96 at most)
  uint32_t const in0 = static_cast<uint32_t>(sizes) * 0x01010101u;
  uint32_t const in1 = static_cast<uint32_t>(sizes >> 32) * 0x01010101u + (in0 >> 24) * 0x01010101u;
  uint32_t const ex0 = in0 << 8, ex1 = __builtin_amdgcn_alignbit(in1, in0, 24);
  uint32_t const sum = in1 >> 24;
  uint32_t total;
  uint32_t const before = block_exclusive_scan_lds<kNormThreads>(sum, lds.scan, &total);
  if (lds.bracket != 0u || total > static_cast<uint32_t>(kStageBytes)) {
    lds_barrier();  // (everybody has read that)
    write_tile(lds, tile, gridDim.x, col, first, n, t, tile_offset, tile_row, out_chars, out_offsets, offsets_are_int64, tid);
    return;
  }
  {
    uint32_t const both = before * 0x00010001u;
    auto const two      = [&](uint32_t v, uint32_t which) { return __builtin_amdgcn_perm(0u, v, which) + both; };
    *reinterpret_cast<uint4*>(&lds.prefix[kNormItems * tid]) =
      make_uint4(two(ex0, 0x0c010c00u), two(ex0, 0x0c030c02u), two(ex1, 0x0c010c00u), two(ex1, 0x0c030c02u));
    if (tid == kNormThreads - 1) lds.prefix[kNormTile] = static_cast<uint16_t>(before + sum);
  }
  uint8_t* const dst  = out_chars + base;
  uint32_t const lead = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst) & 3u);
  uint32_t const o    = lead + before;
  if (!any_long) {
    place_short(reinterpret_cast<uint8_t*>(lds.staged), o, sum, [&](int j) { return text[j] & 0xFFFFFFu; }, [&](int j) { return text[j] >> 24; });
  } else {
    // every string (zero padded) is or-ed into the aligned dwords it falls into; the buffer was cleared, and what the
    // neighbours put into a shared dword is theirs
#pragma unroll
    for (int j = 0; j < kNormItems; ++j) {
      uint32_t const at  = o + (((j < 4 ? ex0 : ex1) >> (8 * (j & 3))) & 0xFFu);
      uint32_t* const to = lds.staged + (at >> 2);
      uint64_t const v   = static_cast<uint64_t>(text[j] & 0xFFFFFFu) << (8u * (at & 3u));
      atomicOr(to, static_cast<uint32_t>(v));
      atomicOr(to + 1, static_cast<uint32_t>(v >> 32));
    }
    uint64_t const ex = (static_cast<uint64_t>(ex1) << 32) | ex0;
#pragma unroll
    for (int k = 0; k < kLongChars; ++k) {
      if (holders[k] == 0) break;
      uint32_t const at  = o + (static_cast<uint32_t>(ex >> at8[k]) & 0xFFu);
      uint32_t const sh  = 8u * (at & 3u);
      uint32_t* const to = lds.staged + (at >> 2);
      uint64_t const a = static_cast<uint64_t>(d0[k]) << sh, b = static_cast<uint64_t>(d1[k]) << sh;
      atomicOr(to, static_cast<uint32_t>(a));
      atomicOr(to + 1, static_cast<uint32_t>(a >> 32) | static_cast<uint32_t>(b));
      if (ballot64((b >> 32) != 0) != 0) atomicOr(to + 2, static_cast<uint32_t>(b >> 32));
    }
  }
  lds_barrier();
  store_staged(lds.staged, dst, lead, total);
  tile_rows.place(col, first, t0, base, lds.prefix, out_offsets, offsets_are_int64);
}

// The same for a column of many tiles, a wavefront a tile as in normalize_count_tiles_kernel: in steps of 512 bytes, whose
// output is laid out in the wavefront's own part of LDS; the line that a step leaves unfinished is the next one's first.
// Tiles that are not for this kernel are left for the workgroup to do together at the end.
// What bounds it is vector instructions, the reads and or-writes of LDS beside them.  Longer characters are taken by fours
// of bytes, two at most in each, with 32-bit arithmetic only; one-byte characters are placed in pairs; a row's place comes
// from the lane that its first byte is with, not from a list of all places.  A step stores whole lines
// (of dwords: 2 to 4 % slower).  766 MB of mixed text 1250 -> 883 to 927 us (traced, as the call then takes 1209 us and more; without
// a trace 1125); a call with a workgroup a tile and with this: 17 MB mixed 73.9 and 76.1 us, ASCII 68.0 and 63.3, 34 MB 105 and 94, 92.3 and 70.8, 134 MB mixed 296 and 235.
constexpr int kStep       = kWave * kNormItems;  // input bytes of a step
constexpr int kStepBytes  = 4 * kStep;           // of output; a tile with more in a step is left
constexpr int kLine       = 128;                 // bytes; a step stores whole lines only
constexpr int kStepWords  = (kStepBytes + kLine) / 4 + 4;
union WriteLds {
  struct {
    alignas(16) uint32_t raw[kTileWaves][kRawWords];
    alignas(16) uint32_t staged[kTileWaves][kStepWords];
    uint32_t third[kTileWaves][4][kWave];  // the last four bytes of strings of more than eight
  };
  NormLds<true> tile;
};
__global__ void __launch_bounds__(kNormThreads, 6) normalize_write_tiles_kernel(ColView col, int64_t first, int64_t n, uint32_t tiles, NormTables t,
                                                                             const uint64_t* __restrict__ tile_offset,
                                                                             const int32_t* __restrict__ tile_row, uint8_t* __restrict__ out_chars,
                                                                             void* __restrict__ out_offsets, int offsets_are_int64)
{
  __shared__ WriteLds lds;
  __shared__ uint32_t ascii[256];
  __shared__ uint32_t left[kTileWaves];  // the tiles left for the end
  uint32_t const wave  = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = lane_id();
  uint32_t const tile0 = blockIdx.x * kTileWaves, tile = tile0 + wave;
  int64_t const t0     = static_cast<int64_t>(tile) * kNormTile;
  const uint8_t* const chars = col.chars + first;
  uint32_t const mis         = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(chars - kRawBefore) & 15u);
  uint32_t* const raw        = lds.raw[wave];
  uint32_t* const staged     = lds.staged[wave];
  uint32_t const table_entry = t.ascii[threadIdx.x];
  bool const third           = lane < kRawWords / 4 - 2 * kWave;
  uint4 v[3];
  int64_t row = 0, row_end = 0;  // the lane's row, of those that begin in the tile
  uint32_t row_at = ~0u;         // where in the tile
  auto const look_up = [&]() {
    row_at = row < row_end ? static_cast<uint32_t>(col.off(row) - first - t0) : ~0u;
  };
  if (tile < tiles) {
    const uint4* const block = reinterpret_cast<const uint4*>(chars + t0 - kRawBefore - mis) + lane;
    if (tile_is_inside(t0, n)) {
      v[0] = load_stream(block);
      v[1] = load_stream(block + kWave);
      if (third) v[2] = load_stream(block + 2 * kWave);
    } else {
      int64_t const p = t0 - kRawBefore - mis + 16 * static_cast<int64_t>(lane);
      v[0]            = load_within(block, p, n);
      v[1]            = load_within(block + kWave, p + 16 * kWave, n);
      if (third) v[2] = load_within(block + 2 * kWave, p + 32 * kWave, n);
    }
    // the rows that start in this tile end where the next tile's begin (the last tile also takes the end of the last row)
    row     = static_cast<int64_t>(tile_row[tile]) + lane;
    row_end = tile + 1 == tiles ? static_cast<int64_t>(col.size) + 1 : static_cast<int64_t>(tile_row[tile + 1]);
    look_up();
  }
  ascii[threadIdx.x] = table_entry;
  for (int i = lane; i < kStepWords / 4; i += kWave) reinterpret_cast<uint4*>(staged)[i] = make_uint4(0u, 0u, 0u, 0u);
  lds_barrier();
  bool marked = false;
  if (tile < tiles) {
    reinterpret_cast<uint4*>(raw)[lane]         = v[0];
    reinterpret_cast<uint4*>(raw)[lane + kWave] = v[1];
    if (third) reinterpret_cast<uint4*>(raw)[lane + 2 * kWave] = v[2];
    wave_lds_sync();
    uint64_t const base  = tile_offset[tile];
    uint8_t* const dst   = out_chars + base;
    uint32_t const lead  = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(dst) & (kLine - 1));
    uint32_t* const dw   = reinterpret_cast<uint32_t*>(dst - lead);
    uint32_t const shift = 8u * (mis & 3u);
    uint32_t words       = 0;     // dwords of the tile's lines that are in memory
    uint32_t in_first    = lead;  // bytes of the buffer's first line that are there already
    // dword w of the buffer, of the bytes [from, to) that are the tile's
    auto const put = [&](uint32_t w, uint32_t d, uint32_t from, uint32_t to) {
      if (4u * w >= from && 4u * w + 4u <= to) {
        store_stream(dw + words + w, d);
      } else {
        for (uint32_t b = max(4u * w, from); b < min(4u * w + 4u, to); ++b)
          reinterpret_cast<uint8_t*>(dw + words)[b] = static_cast<uint8_t>(d >> (8u * (b & 3u)));
      }
    };
    uint32_t done        = 0;     // bytes that the steps before produced
    bool const opened    = t.tokens > 0 && ballot64(opener_before(raw, lane, mis)) != 0;
    const uint32_t* own_raw = raw + ((mis + kRawBefore) >> 2) + 2 * lane;
    marked                  = opened;
#pragma unroll 1
    for (uint32_t from = 0; from < kNormTile && !marked; from += kStep, own_raw += kStep / 4) {
      uint32_t const r0 = own_raw[0], r1 = own_raw[1], r2 = own_raw[2], r3 = own_raw[3];
      uint32_t const own[3] = {__builtin_amdgcn_alignbit(r1, r0, shift), __builtin_amdgcn_alignbit(r2, r1, shift), __builtin_amdgcn_alignbit(r3, r2, shift)};
      uint32_t text[kNormItems];
#pragma unroll
      for (int j = 0; j < kNormItems; ++j) text[j] = ascii[(own[j / 4] >> (8 * (j & 3))) & 0xFFu];
      // the sizes of the positions, a byte each
      auto const top_bytes = [](uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
        return __builtin_amdgcn_perm(b, a, 0x0c0c0703u) | __builtin_amdgcn_perm(d, c, 0x07030c0cu);
      };
      uint32_t sizes[2] = {top_bytes(text[0], text[1], text[2], text[3]), top_bytes(text[4], text[5], text[6], text[7])};
      uint32_t const leads[2] = {own[0] & (own[0] << 1) & 0x80808080u, own[1] & (own[1] << 1) & 0x80808080u};  // bit 7 of the bytes >= 0xC0
      bool const any_long = ballot64((leads[0] | leads[1]) != 0u) != 0;
      bool other          = t.tokens > 0 && (has_byte(own[0], '[') || has_byte(own[1], '['));
      // up to two longer characters in each four bytes: text has no more
      uint32_t d0[4] = {}, d1[4] = {}, at8[4] = {};
      uint64_t holders[4] = {};
      // Strings of more than eight bytes, those of most Hangul syllables in lower case: their last four go through LDS to a pass of their
      // own.  (Left for the workgroup as before, 80 MB of Korean text took 377 us, with a workgroup a tile 369, and takes 238; in
      // registers, or with a branch for each of the four, other text took 1 to 10 % longer.)
      bool any_wide       = false;
      if (any_long) {
        uint4 e[4];
        uint32_t flags = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          uint32_t const all = leads[k / 2], l = k & 1 ? all & (all - 1u) : all;
          holders[k]         = ballot64(l != 0u);
          e[k]               = make_uint4(0u, 0u, 0u, 0u);
          if (holders[k] != 0) {
            at8[k]           = static_cast<uint32_t>(__builtin_ctz(l | 0x80000000u)) & 24u;  // 8 * position
            uint32_t const w = __builtin_amdgcn_alignbit(own[k / 2 + 1], own[k / 2], at8[k]);
            if (l != 0u) e[k] = t.bmp[0x10000u + decode_short(w)];
            bool const four = l != 0u && (w & 0xFFu) >= 0xF0u;
            if (ballot64(four) != 0) {  // (seldom)
              if (four) {
                e[k].w = wide_string(w, t, e[k].x, e[k].y, e[k].z);
                if (e[k].w > 8u || e[k].x == 0x205B20u) e[k].w |= kNotShort;
              }
            }
          }
          if (k & 1) flags |= l & (l - 1u);
        }
        flags |= e[0].w | e[1].w | e[2].w | e[3].w;
        if (ballot64((flags & (kNotShort | 0x808080u)) != 0u) != 0) {  // (seldom)
          // (read from the table once more: whole entries above are 7 to 10 % of other text's time)
          any_wide = true;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            uint32_t const more  = leads[k / 2] & (leads[k / 2] - 1u), w = __builtin_amdgcn_alignbit(own[k / 2 + 1], own[k / 2], at8[k]);
            bool const not_short = (e[k].w & kNotShort) != 0u;
            e[k].w &= 0xFFu;
            // (" [ ": an over-long '[')
            other = other || (more & (more - 1u)) != 0u || (not_short && (e[k].w <= 8u || (w & 0xFFu) >= 0xF0u));
            lds.third[wave][k][lane] = not_short ? t.bmp[0x10000u + decode_short(w)].z : 0u;
          }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          d0[k] = e[k].x;
          d1[k] = e[k].y;
          sizes[k / 2] += e[k].w << at8[k];
        }
      }
      // where each position's bytes begin in the lane's: the sums of the sizes before it (88 at most)
      uint32_t const in0 = sizes[0] * 0x01010101u;
      uint32_t const in1 = sizes[1] * 0x01010101u + (in0 >> 24) * 0x01010101u;
      uint32_t const ex0 = in0 << 8, ex1 = __builtin_amdgcn_alignbit(in1, in0, 24);
      uint32_t const sum    = in1 >> 24;
      uint32_t const incl   = wave_inclusive_scan(sum);
      uint32_t const total  = wave_bcast(incl, kWave - 1);
      uint32_t const before = incl - sum;
      if (ballot64(other) != 0 || total > static_cast<uint32_t>(kStepBytes)) {
        marked = true;
        break;
      }
      // the rows that begin in the step (the end of the last row may lie behind the last tile's last byte)
      uint32_t const row_limit = from + kStep == kNormTile ? kNormTile + 1u : from + kStep;
      while (true) {
        bool const here = row_at >= from && row_at < row_limit;
        if (ballot64(here) != 0) {
          uint32_t const local = row_at - from;
          int const source     = static_cast<int>(local >> 1) & ~3;  // 4 * (local / 8)
          uint32_t const of0   = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(source, static_cast<int>(ex0)));
          uint32_t const of1   = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(source, static_cast<int>(ex1)));
          uint32_t const lanes = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(source, static_cast<int>(before)));
          uint32_t const in    = ((local & 4u ? of1 : of0) >> (8u * (local & 3u))) & 0xFFu;
          if (here) {
            uint64_t const at = base + done + (local >= static_cast<uint32_t>(kStep) ? total : lanes + in);
            if (offsets_are_int64) static_cast<int64_t*>(out_offsets)[row] = static_cast<int64_t>(at);
            else static_cast<int32_t*>(out_offsets)[row] = static_cast<int32_t>(at);
          }
        }
        if (wave_bcast(row_at, kWave - 1) >= row_limit) break;
        row += kWave;  // (more than 64 rows)
        look_up();
      }
      // the one-byte characters in pairs: every string (zero padded) is or-ed into the aligned dwords it falls into; the
      // buffer holds zeros, and what the neighbours put into a shared dword is theirs
      uint32_t const o = in_first + before;
      uint64_t pair[4];
      uint32_t sixes = 0;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        uint32_t const a = text[2 * p], b = text[2 * p + 1];
        pair[p] = (static_cast<uint64_t>(b & 0xFFFFFFu) << ((a >> 21) & 0x18u)) | (a & 0xFFFFFFu);
        sixes |= static_cast<uint32_t>(pair[p] >> 32);
      }
      bool const any_six = ballot64(sixes > 0xFFu) != 0;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        // (a longer character may stand in front of the second: the place is counted from there)
        uint32_t const second = ((p < 2 ? ex0 : ex1) >> (16 * (p & 1) + 8)) & 0xFFu;
        uint32_t const at     = o + second - (text[2 * p] >> 24);
        uint32_t const sh     = 8u * (at & 3u);
        uint32_t* const to    = staged + (at >> 2);
        uint64_t const both   = pair[p] << sh;
        atomicOr(to, static_cast<uint32_t>(both));
        atomicOr(to + 1, static_cast<uint32_t>(both >> 32));
        if (any_six) atomicOr(to + 2, (static_cast<uint32_t>(pair[p] >> 32) >> 8) >> (24u - sh));
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (holders[k] == 0) continue;
        uint32_t const at   = o + (((k < 2 ? ex0 : ex1) >> at8[k]) & 0xFFu);
        uint32_t const sh   = 8u * (at & 3u);
        uint32_t* const to  = staged + (at >> 2);
        uint64_t const both = ((static_cast<uint64_t>(d1[k]) << 32) | d0[k]) << sh;
        uint32_t const past = (d1[k] >> 8) >> (24u - sh);
        atomicOr(to, static_cast<uint32_t>(both));
        atomicOr(to + 1, static_cast<uint32_t>(both >> 32));
        if (ballot64(past != 0u) != 0) atomicOr(to + 2, past);
      }
      if (any_wide) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          uint32_t const at    = o + (((k < 2 ? ex0 : ex1) >> at8[k]) & 0xFFu) + 8u;
          uint64_t const third = static_cast<uint64_t>(lds.third[wave][k][lane]) << (8u * (at & 3u));
          atomicOr(staged + (at >> 2), static_cast<uint32_t>(third));
          atomicOr(staged + (at >> 2) + 1, static_cast<uint32_t>(third >> 32));
        }
      }
      wave_lds_sync();
      // the whole lines to memory, zeros in their place; the unfinished one to the front
      uint32_t const end = in_first + total, full = end / kLine * (kLine / 4);
      uint32_t const rest = lane < kLine / 4 ? staged[full + lane] : 0u;
      if (words != 0 || lead == 0) {
        for (uint32_t w = lane; w < full; w += kWave) {
          store_stream(dw + words + w, staged[w]);
          staged[w] = 0u;
        }
      } else {  // (the tile's first line has bytes of the tile before)
        for (uint32_t w = lane; w < full; w += kWave) {
          put(w, staged[w], lead, 4u * full);
          staged[w] = 0u;
        }
      }
      wave_lds_sync();
      if (lane < kLine / 4) {
        staged[full + lane] = 0u;
        staged[lane]        = rest;
      }
      wave_lds_sync();
      words += full;
      in_first = end % kLine;
      done += total;
    }
    if (!marked && lane < kLine / 4) put(lane, staged[lane], words == 0 ? lead : 0u, in_first);
    if (marked) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // what has been written is there before other wavefronts write it anew
  }
  if (lane == 0) left[wave] = marked ? 1u : 0u;
  lds_barrier();
  if (none_left(left)) return;
#pragma unroll 1
  for (int k = 0; k < kTileWaves; ++k) {
    if (__builtin_amdgcn_readfirstlane(static_cast<int>(left[k])) == 0) continue;
    write_tile(lds.tile, tile0 + k, tiles, col, first, n, t, tile_offset, tile_row, out_chars, out_offsets, offsets_are_int64, same_again(threadIdx.x));
    lds_barrier();
  }
}

struct TileBytes {
  const uint32_t* counts;
  __device__ uint64_t operator()(int64_t i) const { return counts[i]; }
};
// The bytes of the result, for the host.
struct TellBytes {
  uint64_t* host;
  HostPost post;
  __device__ void operator()(uint64_t total) const
  {
    host[0] = total;
    post.send();
  }
};

// ------------------------------------------------------------------ host: tables and tokens
void append_utf8(std::string& s, uint32_t cp)
{
  if (cp < 0x80u) {
    s.push_back(static_cast<char>(cp));
  } else if (cp < 0x800u) {
    s.push_back(static_cast<char>(0xC0u | (cp >> 6)));
    s.push_back(static_cast<char>(0x80u | (cp & 0x3Fu)));
  } else if (cp < 0x10000u) {
    s.push_back(static_cast<char>(0xE0u | (cp >> 12)));
    s.push_back(static_cast<char>(0x80u | ((cp >> 6) & 0x3Fu)));
    s.push_back(static_cast<char>(0x80u | (cp & 0x3Fu)));
  } else {
    s.push_back(static_cast<char>(0xF0u | ((cp >> 18) & 0x07u)));
    s.push_back(static_cast<char>(0x80u | ((cp >> 12) & 0x3Fu)));
    s.push_back(static_cast<char>(0x80u | ((cp >> 6) & 0x3Fu)));
    s.push_back(static_cast<char>(0x80u | (cp & 0x3Fu)));
  }
}

// cudf::strings::to_lower of one string (cpp/src/strings/case.cu:142-148: code points above U+FFFF stay).
// Bytes that are not well-formed UTF-8 are copied as they are.
std::string to_lower_bmp(std::string const& in)
{
  std::string out;
  size_t i = 0;
  auto cont = [&](size_t k) { return k < in.size() && (static_cast<uint8_t>(in[k]) & 0xC0u) == 0x80u; };
  while (i < in.size()) {
    uint32_t const b0 = static_cast<uint8_t>(in[i]);
    uint32_t cp       = b0;
    size_t len        = 1;
    if (b0 >= 0xC2u && b0 < 0xE0u && cont(i + 1)) {
      cp  = ((b0 & 0x1Fu) << 6) | (static_cast<uint8_t>(in[i + 1]) & 0x3Fu);
      len = 2;
    } else if (b0 >= 0xE0u && b0 < 0xF0u && cont(i + 1) && cont(i + 2)) {
      cp  = ((b0 & 0x0Fu) << 12) | ((static_cast<uint8_t>(in[i + 1]) & 0x3Fu) << 6) | (static_cast<uint8_t>(in[i + 2]) & 0x3Fu);
      len = 3;
    } else if (b0 >= 0x80u) {
      len = 1;
      cp  = 0xFFFFFFFFu;  // not a BMP character: copied
      if (b0 >= 0xF0u && cont(i + 1) && cont(i + 2) && cont(i + 3)) len = 4;
    }
    const uint32_t(*row)[4] = nullptr;
    if (cp <= 0xFFFFu) {
      auto const* end = kLowerCase + sizeof(kLowerCase) / sizeof(kLowerCase[0]);
      auto const* it  = std::lower_bound(kLowerCase, end, cp, [](const uint32_t(&r)[4], uint32_t v) { return r[0] < v; });
      if (it != end && (*it)[0] == cp) row = it;
    }
    if (row) {
      for (int k = 1; k < 4; ++k)
        if ((*row)[k]) append_utf8(out, (*row)[k]);
    } else {
      out.append(in, i, len);
    }
    i += len;
  }
  return out;
}

}  // namespace
}  // namespace nvtext_amd

extern "C" {

nvtext_amd_status nvtext_amd_character_normalizer_create(int32_t do_lower_case, const nvtext_amd_strings_column* special_tokens, void* stream_,
                                                         const nvtext_amd_allocator* mr, nvtext_amd_character_normalizer** out)
{
  using namespace nvtext_amd;
  EntryScope const entry("nvtext_amd_character_normalizer_create");
  if (!out) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null argument");
  *out               = nullptr;
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  std::vector<std::string> tokens;
  if (special_tokens && special_tokens->size > 0) {
    // cpp/src/text/normalize.cu:227-228
    if (special_tokens->null_count > 0) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "special tokens should not have nulls");
    int32_t const count = special_tokens->size;
    size_t const ow     = special_tokens->offsets_is_int64 ? 8 : 4;
    std::vector<uint8_t> h_off((static_cast<size_t>(count) + 1) * ow);
    const uint8_t* d_off = static_cast<const uint8_t*>(special_tokens->offsets) + static_cast<size_t>(special_tokens->offset) * ow;
    NVTEXT_HIP_TRY(hipMemcpyAsync(h_off.data(), d_off, h_off.size(), hipMemcpyDeviceToHost, stream));
    NVTEXT_HIP_TRY(hipStreamSynchronize(stream));
    auto off_at = [&](int32_t i) -> int64_t {
      if (ow == 8) {
        int64_t v;
        std::memcpy(&v, h_off.data() + static_cast<size_t>(i) * 8, 8);
        return v;
      }
      int32_t v;
      std::memcpy(&v, h_off.data() + static_cast<size_t>(i) * 4, 4);
      return v;
    };
    int64_t const first = off_at(0), last = off_at(count);
    if (last < first) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "special token offsets are not monotone");
    std::string pool(static_cast<size_t>(last - first), '\0');
    if (!pool.empty()) {
      NVTEXT_HIP_TRY(hipMemcpyAsync(&pool[0], special_tokens->chars + first, pool.size(), hipMemcpyDeviceToHost, stream));
      NVTEXT_HIP_TRY(hipStreamSynchronize(stream));
    }
    for (int32_t i = 0; i < count; ++i) tokens.emplace_back(pool, static_cast<size_t>(off_at(i) - first), static_cast<size_t>(off_at(i + 1) - off_at(i)));
    // cpp/src/text/normalize.cu:230-235: sorted by bytes first, lower-cased afterwards
    std::sort(tokens.begin(), tokens.end(), [](std::string const& a, std::string const& b) {
      int const c = std::memcmp(a.data(), b.data(), std::min(a.size(), b.size()));
      return c != 0 ? c < 0 : a.size() < b.size();
    });
    if (do_lower_case)
      for (auto& tk : tokens) tk = to_lower_bmp(tk);
  }

  // dense tables from the generated runs; the Hangul syllables decompose by arithmetic (The Unicode Standard, 3.12)
  std::vector<uint32_t> entries(kCodepoints, kDefaultEntry);
  std::vector<uint64_t> second(kCodepoints, 0);
  for (auto const& run : kCodepointRuns) std::fill(entries.begin() + run[0], entries.begin() + run[0] + run[1], run[2]);
  for (auto const& pair : kCodepointSecond) second[static_cast<size_t>(pair[0])] = pair[1];
  for (uint32_t s = 0; s < 11172u; ++s) {
    uint32_t const lead = 0x1100u + s / 588u, vowel = 0x1161u + (s % 588u) / 28u, trail = s % 28u;
    entries[0xAC00u + s] = (5u << 24) | (1u << 23) | lead;
    second[0xAC00u + s]  = (static_cast<uint64_t>(vowel) << 32) | (trail ? 0x11A7u + trail : 0u);
  }

  // the slots of the one-byte code points, decided here once (the rules of slots_of)
  uint32_t ascii[256] = {};
  for (uint32_t cp = 0; cp < 128u; ++cp) {
    uint32_t const e = entries[cp], cat = (e >> 24) & 7u;
    uint32_t d       = 0;
    if (!(cat == kRemove || (do_lower_case && cat == kRemoveIfLower))) {
      uint32_t const repl = (do_lower_case || cat == kReplace) ? (e & 0x1FFFFFu) : cp;
      uint32_t const r0   = repl ? repl : cp;
      d                   = (cat == kPad || (do_lower_case && cat == kPadIfLower)) ? (0x20u | (r0 << 8) | (0x20u << 16) | (3u << 24)) : (r0 | (1u << 24));
    }
    ascii[cp] = d;
  }

  // the finished slots of the Basic Multilingual Plane (the rules of slots_of, run here once per code point)
  std::vector<uint4> bmp(2 * 0x10000);
  std::vector<uint8_t> sizes(0x10000);
  {
    NormTables const host_tables{nullptr, nullptr, nullptr, entries.data(), second.data(), nullptr, nullptr, 0, do_lower_case ? 1 : 0};
    for (uint32_t cp = 0; cp < 0x10000u; ++cp) {
      uint32_t s0, s1, s2;
      slots_of(cp, host_tables, s0, s1, s2);
      bmp[cp]   = make_uint4(s0, s1, s2, bytes_of(s0) + bytes_of(s1) + bytes_of(s2));
      sizes[cp] = static_cast<uint8_t>(bmp[cp].w);
      uint32_t d0, d1, d2;
      slots_to_string(s0, s1, s2, d0, d1, d2);
      bmp[0x10000 + cp] = make_uint4(d0, d1, d2, bmp[cp].w | (bmp[cp].w > 8u || d0 == 0x205B20u ? kNotShort : 0u));
    }
  }

  auto* obj      = new nvtext_amd_character_normalizer();
  obj->do_lower  = do_lower_case ? 1 : 0;
  obj->tokens    = static_cast<int32_t>(tokens.size());
  auto fail_with = [&](hipError_t e) {
    nvtext_amd_character_normalizer_destroy(obj);
    return fail(e == hipErrorOutOfMemory ? NVTEXT_AMD_ALLOC_FAILED : NVTEXT_AMD_DEVICE_ERROR, hipGetErrorString(e));
  };
  obj->store.bind(mr, stream);
  std::vector<int32_t> token_offsets(tokens.size() + 1, 0);
  std::string token_chars;
  for (size_t i = 0; i < tokens.size(); ++i) {
    token_chars += tokens[i];
    if (token_chars.size() > 0x7FFFFFFFull) {
      nvtext_amd_character_normalizer_destroy(obj);
      return fail(NVTEXT_AMD_OVERFLOW, "special tokens too large");
    }
    token_offsets[i + 1] = static_cast<int32_t>(token_chars.size());
  }
  hipError_t e = hipGetDevice(&obj->device);
  if (e != hipSuccess) return fail_with(e);
  bool ok = obj->store.allocate(&obj->ascii, 256) && obj->store.allocate(&obj->bmp, bmp.size()) &&
            obj->store.allocate(&obj->sizes, sizes.size()) && obj->store.allocate(&obj->entries, entries.size()) && obj->store.allocate(&obj->second, second.size());
  if (ok && !tokens.empty())
    ok = obj->store.allocate(&obj->token_offset, token_offsets.size()) && obj->store.allocate(&obj->token_chars, token_chars.size() + 8);
  if (!ok) return fail_with(hipErrorOutOfMemory);
  e = hipMemcpyAsync(obj->ascii, ascii, sizeof(ascii), hipMemcpyHostToDevice, stream);
  if (e == hipSuccess) e = hipMemcpyAsync(obj->bmp, bmp.data(), bmp.size() * sizeof(uint4), hipMemcpyHostToDevice, stream);
  if (e == hipSuccess) e = hipMemcpyAsync(obj->sizes, sizes.data(), sizes.size(), hipMemcpyHostToDevice, stream);
  if (e == hipSuccess) e = hipMemcpyAsync(obj->entries, entries.data(), entries.size() * sizeof(uint32_t), hipMemcpyHostToDevice, stream);
  if (e == hipSuccess) e = hipMemcpyAsync(obj->second, second.data(), second.size() * sizeof(uint64_t), hipMemcpyHostToDevice, stream);
  if (e == hipSuccess && !tokens.empty())
    e = hipMemcpyAsync(obj->token_offset, token_offsets.data(), token_offsets.size() * sizeof(int32_t), hipMemcpyHostToDevice, stream);
  token_chars.append(8, '\0');
  if (e == hipSuccess && !tokens.empty()) e = hipMemcpyAsync(obj->token_chars, token_chars.data(), token_chars.size(), hipMemcpyHostToDevice, stream);
  hipError_t const synced = hipStreamSynchronize(stream);  // the host copies die at return
  if (e == hipSuccess) e = synced;
  if (e != hipSuccess) return fail_with(e);
  *out = obj;
  return NVTEXT_AMD_SUCCESS;
}

void nvtext_amd_character_normalizer_destroy(nvtext_amd_character_normalizer* normalizer)
{
  delete normalizer;  // the store hands the tables back
}

nvtext_amd_status nvtext_amd_normalize_characters(const nvtext_amd_strings_column* input, const nvtext_amd_character_normalizer* normalizer,
                                                  void* stream_, const nvtext_amd_allocator* mr_, nvtext_amd_strings_result* out)
{
  using namespace nvtext_amd;
  EntryScope const entry("nvtext_amd_normalize_characters");
  if (!input || !normalizer || !out) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null argument");
  *out = nvtext_amd_strings_result{};
  if (input->size < 0 || input->null_count < 0 || input->null_count > input->size) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "invalid column sizes");
  if (input->null_count > 0 && !input->null_mask) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null_count > 0 requires a null mask");
  int device = 0;
  NVTEXT_HIP_TRY(hipGetDevice(&device));
  if (device != normalizer->device) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "the normalizer belongs to another device");
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  Mr mr{mr_, stream};
  int32_t const rows = input->size;
  if (rows == 0) return NVTEXT_AMD_SUCCESS;  // normalize.cu:497: the empty strings column
  if (!input->offsets) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "offsets missing");

  // normalize.cu:499-501: the byte range of the view.  A column of few rows is probably small, and then launches and waits
  // are most of the call: the sizes of the tiles' outputs are put on the stream as well, for a column of up to
  // kSmallRowBytes bytes a row and kSmallBytes in all, before the host knows how many bytes there are; one wait instead of
  // two.  Where there are more these kernels leave at once.  (61 rows of 300 bytes: 74 -> 32 us)
  ColView const view = make_view(*input);
  NormTables const tables{normalizer->ascii, normalizer->bmp, normalizer->sizes, normalizer->entries, normalizer->second, normalizer->token_chars, normalizer->token_offset, normalizer->tokens,
                          normalizer->do_lower};
  uint64_t* const scalars = host_scalars();  // pinned words that kernels write for the host (nullptr: copy instead)
  bool small              = scalars && input->chars && rows <= kSmallRows;
  int64_t const small_bytes = small ? std::min(std::max(static_cast<int64_t>(rows) * kSmallRowBytes, kSmallLeast), kSmallBytes) : 0;
  size_t const small_tiles  = static_cast<size_t>(small_bytes / kNormTile + 1);
  size_t const small_temp_bytes[3] = {small_tiles * sizeof(uint32_t), small_tiles * sizeof(uint64_t), small_tiles * sizeof(int32_t)};
  TempParts<3> const small_temps(mr, small_temp_bytes, small);
  if (small && !small_temps.ok()) return fail(NVTEXT_AMD_ALLOC_FAILED, "temporary allocation failed");
  int64_t first = 0, last = 0;
  uint64_t total = 0;
  if (scalars) {
    HostPost const post = new_post();
    if (small) {
      unsigned const grid = static_cast<unsigned>(std::min<size_t>(small_tiles, static_cast<size_t>(device_cus()) * 16));
      hipLaunchKernelGGL(normalize_count_small_kernel, dim3(grid), dim3(kNormThreads), 0, stream, view, small_bytes, tables, small_temps.part<uint32_t>(0),
                         small_temps.part<int32_t>(2));
      hipLaunchKernelGGL(normalize_finish_kernel, dim3(1), dim3(kFinishThreads), 0, stream, view, small_bytes, small_temps.part<uint32_t>(0),
                         small_temps.part<uint64_t>(1), scalars, post);
    } else {
      launch_read_two_offsets(input->offsets, input->offsets_is_int64 != 0, input->offset, static_cast<int64_t>(input->offset) + rows, scalars, post, stream);
    }
    NVTEXT_HIP_TRY(hipGetLastError());
    NVTEXT_HIP_TRY(wait_for_post(post, stream));
    first = static_cast<int64_t>(scalars[0]);
    last  = static_cast<int64_t>(scalars[1]);
    total = scalars[2];
  } else {
    size_t const ow      = input->offsets_is_int64 ? 8 : 4;
    const uint8_t* d_off = static_cast<const uint8_t*>(input->offsets) + static_cast<size_t>(input->offset) * ow;
    int64_t ends[2]      = {0, 0};
    int32_t ends32[2]    = {0, 0};
    for (int k = 0; k < 2; ++k) {
      void* host = ow == 8 ? static_cast<void*>(&ends[k]) : static_cast<void*>(&ends32[k]);
      NVTEXT_HIP_TRY(hipMemcpyAsync(host, d_off + (k ? static_cast<size_t>(rows) * ow : 0), ow, hipMemcpyDeviceToHost, stream));
    }
    NVTEXT_HIP_TRY(hipStreamSynchronize(stream));
    first = ow == 8 ? ends[0] : ends32[0];
    last  = ow == 8 ? ends[1] : ends32[1];
  }
  if (last < first) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "offsets are not monotone");
  int64_t const n = last - first;
  if (n > 0 && !input->chars) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "chars missing");
  small = small && n <= small_bytes;

  auto release = [&](nvtext_amd_status st, const char* msg) {
    nvtext_amd_strings_result_free(out, stream_, mr_);
    return fail(st, msg);
  };
  out->size         = rows;
  out->null_count   = input->null_count;
  out->offsets_size = rows + 1;
  auto allocate_offsets = [&](bool wide) {
    out->offsets_is_int64 = wide ? 1 : 0;
    out->offsets_bytes    = (static_cast<size_t>(rows) + 1) * (wide ? sizeof(int64_t) : sizeof(int32_t));
    out->offsets          = mr.allocate(out->offsets_bytes);
    return out->offsets != nullptr;
  };
  if (input->null_mask) {  // copy_bitmask(input): cpp/src/bitmask/null_mask.cu:381-391
    out->null_mask_bytes = mask_alloc_bytes(rows);
    out->null_mask       = static_cast<uint32_t*>(mr.allocate(out->null_mask_bytes));
    if (!out->null_mask) return release(NVTEXT_AMD_ALLOC_FAILED, "mask allocation failed");
    launch_copy_bitmask(out->null_mask, input->null_mask, input->offset, rows, stream);
  }
  if (n == 0) {  // normalize.cu:504: nothing to normalize, every row is empty
    if (!allocate_offsets(false)) return release(NVTEXT_AMD_ALLOC_FAILED, "result allocation failed");
    launch_fill_u32(static_cast<uint32_t*>(out->offsets), 0u, static_cast<int64_t>(rows) + 1, stream);
    NVTEXT_HIP_TRY_OR(hipGetLastError(), nvtext_amd_strings_result_free(out, stream_, mr_));
    return NVTEXT_AMD_SUCCESS;
  }

  int64_t const tiles = (n + kNormTile - 1) / kNormTile;
  if (tiles > 0x7FFFFFFFll) return release(NVTEXT_AMD_OVERFLOW, "input too large");
  size_t const temp_bytes[4] = {static_cast<size_t>(tiles) * sizeof(uint32_t), (static_cast<size_t>(tiles) + 1) * sizeof(uint64_t),
                                scan_temp_bytes(tiles), static_cast<size_t>(tiles) * sizeof(int32_t)};
  TempParts<4> const temps(mr, temp_bytes, !small);
  if (!small && !temps.ok()) return release(NVTEXT_AMD_ALLOC_FAILED, "temporary allocation failed");
  uint64_t* const tile_offset = small ? small_temps.part<uint64_t>(1) : temps.part<uint64_t>(1);
  int32_t* const tile_row     = small ? small_temps.part<int32_t>(2) : temps.part<int32_t>(3);
  hipError_t e                = hipSuccess;
  if (!small) {
    uint32_t* const tile_bytes = temps.part<uint32_t>(0);
    {
      ProfileScope ps("normalize_count_kernel", stream);
      if (tiles >= kManyTiles) {
        int64_t const grid = (tiles + kTileWaves - 1) / kTileWaves;
        hipLaunchKernelGGL(normalize_count_tiles_kernel, dim3(static_cast<unsigned>(grid)), dim3(kNormThreads), 0, stream, view.chars + first, n,
                           static_cast<uint32_t>(tiles), tables, tile_bytes);
      } else {
        hipLaunchKernelGGL(normalize_count_kernel, dim3(static_cast<unsigned>(tiles)), dim3(kNormThreads), 0, stream, view.chars + first, n, tables,
                           tile_bytes);
      }
    }
    bool const few_tiles = tiles <= kSearchTiles;
    hipLaunchKernelGGL(few_tiles ? normalize_tile_rows_kernel<8> : normalize_tile_rows_kernel<1>, dim3(static_cast<unsigned>((tiles * (few_tiles ? 8 : 1) + 255) / 256)),
                       dim3(256), 0, stream, view, first, tiles, tile_row);
    if (scalars) {
      HostPost const post = new_post();
      device_exclusive_scan(TileBytes{tile_bytes}, tiles, tile_offset, temps.part<uint64_t>(2), stream, TellBytes{scalars, post});
      e = hipGetLastError();
      if (e == hipSuccess) e = wait_for_post(post, stream);
    } else {
      device_exclusive_scan(TileBytes{tile_bytes}, tiles, tile_offset, temps.part<uint64_t>(2), stream, TellNobody{});
      e = hipMemcpyAsync(&total, tile_offset + tiles, sizeof(total), hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipStreamSynchronize(stream);
    }
    if (e != hipSuccess) return release(NVTEXT_AMD_DEVICE_ERROR, hipGetErrorString(e));
    if (scalars) total = scalars[0];
  }
  // int64 offsets from the large-strings threshold on (cpp/include/cudf/strings/detail/strings_children.cuh:164-175)
  if (!allocate_offsets(total >= 0x7FFFFFFFull)) return release(NVTEXT_AMD_ALLOC_FAILED, "result allocation failed");
  out->chars_size = static_cast<int64_t>(total);
  if (total > 0) {
    out->chars_bytes = static_cast<size_t>(total);
    out->chars       = static_cast<char*>(mr.allocate(out->chars_bytes));
    if (!out->chars) return release(NVTEXT_AMD_ALLOC_FAILED, "result allocation failed");
  }
  {
    ProfileScope ps("normalize_write_kernel", stream);
    if (tiles >= kManyTiles) {
      int64_t const grid = (tiles + kTileWaves - 1) / kTileWaves;
      hipLaunchKernelGGL(normalize_write_tiles_kernel, dim3(static_cast<unsigned>(grid)), dim3(kNormThreads), 0, stream, view, first, n,
                         static_cast<uint32_t>(tiles), tables, tile_offset, tile_row, reinterpret_cast<uint8_t*>(out->chars), out->offsets,
                         out->offsets_is_int64);
    } else {
      hipLaunchKernelGGL(normalize_write_kernel, dim3(static_cast<unsigned>(tiles)), dim3(kNormThreads), 0, stream, view, first, n, tables,
                         tile_offset, tile_row, reinterpret_cast<uint8_t*>(out->chars), out->offsets, out->offsets_is_int64);
    }
  }
  e = hipGetLastError();
  if (e != hipSuccess) return release(NVTEXT_AMD_DEVICE_ERROR, hipGetErrorString(e));
  return NVTEXT_AMD_SUCCESS;
}

void nvtext_amd_strings_result_free(nvtext_amd_strings_result* col, void* stream, const nvtext_amd_allocator* mr)
{
  if (!col) return;
  nvtext_amd::Mr m{mr, static_cast<hipStream_t>(stream)};
  m.deallocate(col->offsets, col->offsets_bytes);
  m.deallocate(col->chars, col->chars_bytes);
  m.deallocate(col->null_mask, col->null_mask_bytes);
  *col = nvtext_amd_strings_result{};
}

}  // extern "C"
