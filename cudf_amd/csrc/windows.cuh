// Character windows of a row, shared by minhash and jaccard_index: a wavefront stages a tile of row bytes
// in LDS with aligned 16-byte loads and decides, per byte position, whether a `width`-character window
// starts there and how many bytes it spans
// (cpp/src/text/minhash.cu:120-133, cpp/src/text/jaccard.cu:268-277, cpp/include/cudf/strings/string_view.cuh:67-80).
#pragma once

#include "common.cuh"
#include "murmur.cuh"

#include <type_traits>

namespace nvtext_amd {

constexpr int kWaves     = 4;                  // wavefronts per workgroup
constexpr int kThreads   = kWaves * kWave;     // 256
constexpr int kTile      = 256;                // window starts per wavefront tile
constexpr int kHalo      = 128;                // bytes staged past the tile (windows up to 32 4-byte chars)
constexpr int kCharList  = kTile + kHalo + 8;   // list of a tile's characters: one per staged byte, the end of the last one, padding
constexpr int kTileWords = (kTile + kHalo + 16 + 32) / 4;  // +16 misalignment, +32 for whole blocks and the over-read of the hash tail

// 64-bit hashes: so many are gathered before they meet the parameters, which costs as much for few as for many where it ends
// (the exact products).  What leaves four workgroups to a CU with up to 160 parameters: 20,011 long rows, 128 parameters:
// 352: 2860 us, 416: 2802; with more, three: 448 of them and a wavefront less are 5 to 12 % slower where 416 would do.
constexpr uint32_t kFoldFrom = 416;

// Windows repeat (of 2 KB of ordinary text three in four are different, of 16 KB little more than half), and a hash that
// has been folded once changes no minimum when it is folded again.  Every wavefront keeps the hashes it saw last in a
// small direct-mapped table (of 64-bit hashes, the places that they have among those gathered: 2 KB for 1024 where 512
// hashes took 4) and drops a hash that it finds there; what the table has forgotten is folded again, which
// costs time and nothing else.  Cleared (hashes are never 0) whenever the wavefront begins a part of a row.  As many entries as leave
// six (64-bit hashes: four) workgroups to a CU: 400,000 documents of 2 KB, 256 parameters of 32 bits: 256 entries 8.80 ms,
// 512: 8.45, 1024: 8.17.
constexpr uint32_t kRecentEntries = 1024;
constexpr uint32_t kNoPlace       = kFoldFrom + kTile + 31;
template <typename T>
struct WaveLds {
  alignas(16) uint32_t bytes[kTileWords];
  alignas(16) T hashes[sizeof(T) == 4 ? kTile + 4 : kNoPlace + 1];
  alignas(16) std::conditional_t<sizeof(T) == 4, T, uint16_t> recent[kRecentEntries];
  uint16_t chars[kCharList];  // where the characters of the staged bytes start, in order (see CharMap)
};

// The aligned 16-byte blocks that bytes [at, at + len) lie in, a lane a block (at most 64 of them): fetch() asks for them and does
// not wait, stage() puts them into LDS.  Only blocks that overlap the range are read.
struct TileBytes {
  uint4 block;
  uint32_t mis;  // byte offset of `at` in the first block
  uint32_t blocks;
  __device__ __forceinline__ void fetch(const uint8_t* at, uint32_t len, int lane)
  {
    mis    = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(at) & 15u);
    blocks = (mis + len + 15u) >> 4;
    block  = make_uint4(0u, 0u, 0u, 0u);
    if (static_cast<uint32_t>(lane) < blocks) block = reinterpret_cast<const uint4*>(at - mis)[lane];
  }
  // dst: 16-byte aligned.  *all_ascii: no byte of these blocks has its top bit set (wave-uniform); a byte beyond ASCII next to
  // the range costs the caller its shorter way and nothing else.
  __device__ __forceinline__ void stage(uint32_t* dst, int lane, bool* all_ascii) const
  {
    if (static_cast<uint32_t>(lane) < blocks) reinterpret_cast<uint4*>(dst)[lane] = block;
    *all_ascii = ballot64(((block.x | block.y | block.z | block.w) & 0x80808080u) != 0) == 0;
  }
};

// Stage row bytes [base, base+len), any number of them, into dst (16-byte aligned); returns the byte offset of `base` inside it.
__device__ __forceinline__ uint32_t stage_bytes(const uint8_t* row, int64_t base, uint32_t len, uint32_t* dst, int lane)
{
  const uint8_t* g   = row + base;
  uint32_t const mis = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(g) & 15u);
  const uint4* ap    = reinterpret_cast<const uint4*>(g - mis);
  uint32_t const nb  = (mis + len + 15u) >> 4;
  for (uint32_t i = lane; i < nb; i += kWave) reinterpret_cast<uint4*>(dst)[i] = ap[i];
  return mis;
}

// The characters of the staged bytes of a tile, found by the whole wavefront at once, for tiles that hold bytes beyond
// ASCII.  The reference walks from every window start byte by byte, adding up what each first byte of a character
// says of its length until `width` characters are counted (cpp/include/cudf/strings/string_view.cuh:67-80).  Where
// every character of the staged bytes ends exactly where the next one starts, that sum is the distance from the start
// of character k to the start of character k + width: the starts are listed in LDS, in order, and a lane takes a
// character instead of a byte position, and a window costs two reads of the list.  Other tiles (stray continuation bytes,
// first bytes that promise more than follows) keep the walk.
// A lane looks at eight bytes, by their top bits: which bytes continue a character, and which ought to by the first bytes
// before them.  (As 64-bit masks of a bit a byte, 64 bytes at a time, the same took 300 scalar instructions a tile, of which
// a CU issues one a cycle for its four SIMDs: 2.4 of the 5.2 ms of 1,000,003 rows of 512 bytes, 64-bit hashes, 64 parameters, which
// now take 4.8; jaccard, 100,000 pairs of 1000 bytes 1451 -> 1139 us.)
struct CharMap {
  uint32_t count;    // characters that start in the staged bytes
  uint32_t windows;  // of them, in the tile's window starts (the first `cnt` staged bytes)
  bool exact;        // the list gives every window of the tile its length

  // The top bits of the bytes [from, to) of eight.
  static __device__ __forceinline__ uint64_t tops(int32_t from, int32_t to)
  {
    uint64_t const all = 0x8080808080808080ull;
    uint32_t const low = static_cast<uint32_t>(min(max(from, 0), 8)) * 4u, high = static_cast<uint32_t>(8 - min(max(to, 0), 8)) * 4u;
    return (all << low << low) & (all >> high >> high);
  }
  // Bytes i - n of eight and of the eight before, at i.
  static __device__ __forceinline__ uint64_t moved_up(uint64_t v, uint32_t before, uint32_t n)
  {
    uint32_t const lo = static_cast<uint32_t>(v), hi = static_cast<uint32_t>(v >> 32);
    return static_cast<uint64_t>(__builtin_amdgcn_alignbyte(hi, lo, 4u - n)) << 32 | __builtin_amdgcn_alignbyte(lo, before, 4u - n);
  }
  static __device__ __forceinline__ uint32_t of_lane_below(uint64_t v)  // its upper half; lane 0: 0
  {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v >> 32), 0x138, 0xF, 0xF, true));
  }

  // staged: the tile's bytes in LDS, its first byte at byte offset `mis`; len of them are the row's, the first cnt are
  // window starts; chars: the list (kCharList entries).
  __device__ __forceinline__ void build(const uint32_t* staged, uint32_t mis, uint32_t len, uint32_t cnt, bool reaches_row_end, uint16_t* chars,
                                        int lane)
  {
    static_assert(kTile + kHalo + 15 <= 8 * kWave, "eight bytes a lane");
    int32_t const at  = 8 * lane - static_cast<int32_t>(mis);  // place of the lane's first byte
    uint64_t x        = 0;
    if (at < static_cast<int32_t>(len)) x = reinterpret_cast<const uint64_t*>(staged)[lane];
    uint64_t const here  = tops(-at, static_cast<int32_t>(len) - at);
    uint64_t const x1    = x << 1, x2 = x << 2, x3 = x << 3;  // (only top bits are looked at)
    uint64_t const cont  = x & ~x1 & here;
    uint64_t const start = ~cont & here;
    uint64_t const two   = x & x1 & here, three = two & x2, four = three & x3;  // what begins a character of two bytes and more, ..
    uint64_t const expected = moved_up(two, of_lane_below(two), 1) | moved_up(three, of_lane_below(three), 2) | moved_up(four, of_lane_below(four), 3);
    uint64_t const with     = ballot64(start != 0);
    int const first_lane    = __builtin_ctzll(with | 1ull << 63), last_lane = 63 - __builtin_clzll(with | 1ull);
    // (bytes before the first character of the tile belong to one that began before it)
    uint64_t const before = lane > first_lane ? 0ull : ~start & (start - 1ull);
    bool const wrong      = ((expected ^ cont) & here & ~before) != 0;
    // starts of the lane, and of them in the window starts; those of the lanes before
    uint64_t const in_tile = start & tops(-at, static_cast<int32_t>(cnt) - at);
    uint32_t const n       = static_cast<uint32_t>(__builtin_popcountll(start)) | static_cast<uint32_t>(__builtin_popcountll(in_tile)) << 16;
    uint32_t const upto    = wave_inclusive_scan(n);
    uint32_t const total   = wave_bcast(upto, kWave - 1);
    count                  = total & 0xFFFFu;
    windows                = total >> 16;
    uint32_t to            = (upto & 0xFFFFu) - (n & 0xFFFFu);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if ((start >> (8 * j + 7)) & 1u) chars[to] = static_cast<uint16_t>(at + j);
      to += static_cast<uint32_t>(start >> (8 * j + 7)) & 1u;
    }
    // the last character: where it starts and where it ends by its first byte
    int const top            = 63 - __builtin_clzll(start | 1ull);
    uint32_t const mine      = static_cast<uint32_t>(at + top / 8) | (1u + static_cast<uint32_t>((two >> top & 1u) + (three >> top & 1u) + (four >> top & 1u))) << 16;
    uint32_t const last      = wave_bcast(mine, last_lane);
    uint32_t const last_start = last & 0xFFFFu, last_end = last_start + (last >> 16);
    if (lane == 0) chars[count] = static_cast<uint16_t>(last_end);
    wave_lds_fence();
    // the last one: ends with the row, or, when the row goes on, begins in the last four staged bytes (then every window
    // start of the tile, at least 4 * width bytes before the end of the staged bytes, has its `width` characters listed)
    exact = ballot64(wrong) == 0 && count > 0 && (reaches_row_end ? last_end == len : len - last_start <= 4u);
  }

  // The window that begins with character k (k < windows): whether it counts, where it starts and its bytes.
  // row_start: staged byte 0 is the row's first byte.
  __device__ __forceinline__ bool window(uint32_t k, uint32_t len, bool row_start, int32_t width, const uint16_t* chars, uint32_t* pos,
                                         uint32_t* hlen) const
  {
    uint32_t const first = chars[k];
    *pos                 = first;
    // fewer than `width` characters are left (the staged bytes reach the end of the row): only the row's first position counts
    bool const whole = k + static_cast<uint32_t>(width) <= count;
    *hlen            = (whole ? chars[k + static_cast<uint32_t>(width)] : len) - first;
    return whole || (row_start && first == 0);
  }
};

// Decides whether a window starts at this position and how many bytes it hashes
// (cpp/src/text/minhash.cu:120-133 with cpp/include/cudf/strings/string_view.cuh:67-80).
// `remaining` = row bytes from this position on; `readable` = bytes of them reachable through src
// (the whole rest of the row, or at least 4 * width bytes); `g` = this position in the row itself.
template <typename Src>
__device__ __forceinline__ bool window_at(Src const& src, const uint8_t* g, int64_t remaining, uint32_t readable, bool first, bool all_ascii,
                                          int32_t width, uint32_t* hlen)
{
  if (all_ascii) {
    if (remaining >= width) {
      *hlen = static_cast<uint32_t>(width);
      return true;
    }
    *hlen = static_cast<uint32_t>(remaining);
    return first;
  }
  if (is_utf8_continuation(src.byte(0))) return false;
  uint32_t bytes = 0, j = 0;
  int32_t left = width;
  while (left > 0 && j < readable) {  // byte-wise, as the reference walks
    int const w = bytes_in_utf8_byte(src.byte(j));
    left -= (w != 0);
    bytes += w;
    ++j;
  }
  // Well-formed text has `width` characters within 4 * width bytes.  Bytes that continue no character count for
  // nothing, so a run of them can leave characters to find beyond what src reaches: the walk goes on in the row.
  if (left > 0 && j < remaining) {
    int64_t k = j;
    while (left > 0 && k < remaining) {
      int const w = bytes_in_utf8_byte(g[k]);
      left -= (w != 0);
      bytes += w;
      ++k;
    }
  }
  // a malformed trailing lead byte may declare more bytes than the row holds: clamp to the row
  *hlen = static_cast<uint32_t>(min(static_cast<int64_t>(bytes), remaining));
  return first || left <= 0;
}

// The windows that start in [base, base + cnt) of (the rest of) a row, n bytes from `row` on (cnt <= kTile, 4 * width <= kHalo):
// `hash(src, bytes, h)` of each (arrays of one source and hash or of two, of one length) goes to `sink(valid, h)`, which every
// lane of the wavefront calls together, with arrays of one window per lane or of two (two chains of LDS reads and multiplies
// in flight instead of one).  `bytes` and `chars` are the wavefront's own LDS.  starts: `row` is the row's first byte.  Places
// have 32 bits, which take half the scalar registers and instructions; `beyond` more bytes than n belong to a row that is
// longer.  tile: the row's bytes from base on, tile_length() of them; when they are in LDS, next() may ask for others.  FOUR: sink()
// takes four windows a lane as well, from whole tiles.
__device__ __forceinline__ uint32_t tile_length(int32_t n, int32_t base, uint32_t cnt, int32_t width)
{
  return min(static_cast<uint32_t>(n - base), cnt + static_cast<uint32_t>(width) * 4u);
}
template <typename T, bool FOUR = false, typename Next, typename Hash, typename Sink>
__device__ __forceinline__ void hash_tile_windows(TileBytes& tile, Next&& next, const uint8_t* row, int32_t n, int64_t beyond, bool starts, int32_t base, uint32_t cnt,
                                                  int32_t width, uint32_t* bytes, uint16_t* chars, int lane, Hash const& hash, Sink&& sink)
{
  uint32_t const len = tile_length(n, base, cnt, width);
  uint32_t const mis = tile.mis;
  bool all_ascii;
  tile.stage(bytes, lane, &all_ascii);
  next();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // In a tile of one-byte characters of a row that has `width` bytes and more every window is `width` bytes long: the
  // hash then runs with a length that the compiler knows to be the same in every lane (its loops over the
  // blocks and the tail become scalar branches instead of masked ones).
  bool const plain         = all_ascii && (!starts || n >= width);
  uint32_t const width_all = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(width));
  if (plain) {
    // (the last window of the row ends with it)
    uint32_t const starts_here = min(cnt, len - min(len, width_all - 1u));
    // (a lane beyond the last window hashes what lies there in the tile's LDS: no branch, and one address for both windows)
    static_assert(kTile + kWave + kHalo / 4 + 32 <= 4 * kTileWords);
    uint32_t const here = mis + lane;
    uint32_t q          = 0;
    if constexpr (FOUR) {
      static_assert(kTile == 4 * kWave);
      if (starts_here > 3u * kWave) {
        bool const valid[4]  = {true, true, true, 3 * kWave + lane < starts_here};
        WordSrc const src[4] = {WordSrc(bytes, here), WordSrc(bytes + kWave / 4, here), WordSrc(bytes + 2 * kWave / 4, here), WordSrc(bytes + 3 * kWave / 4, here)};
        T hv[4];
        hash(src, width_all, hv);
        sink(valid, hv);
        q = kTile;
      }
    }
    for (; q + kWave < starts_here; q += 2 * kWave) {
      bool const valid[2]  = {true, q + kWave + lane < starts_here};
      WordSrc const src[2] = {WordSrc(bytes + q / 4, here), WordSrc(bytes + q / 4 + kWave / 4, here)};
      T hv[2];
      hash(src, width_all, hv);
      sink(valid, hv);
    }
    if (q < starts_here) {
      bool const valid[1]  = {q + lane < starts_here};
      WordSrc const src[1] = {WordSrc(bytes + q / 4, here)};
      T hv[1];
      hash(src, width_all, hv);
      sink(valid, hv);
    }
  } else {
    // A tile with longer characters: all of them are found at once, and where they follow one another without a gap
    // a lane takes a character, not a byte, and reads its window's length from the list of characters instead of
    // walking.  (A row shorter than `width` comes here too, whatever its bytes.)
    CharMap map;
    map.exact = false;
    if (!all_ascii) map.build(bytes, mis, len, cnt, base + static_cast<int32_t>(len) == n, chars, lane);
    uint32_t const items = map.exact ? map.windows : cnt;  // characters, or byte positions
    for (uint32_t q = 0; q < items; q += kWave) {
      uint32_t const item = q + lane;
      bool valid[1]       = {false};
      T hv[1]             = {0};
      if (item < items) {
        uint32_t p = item, hlen;
        bool const first = starts && base == 0;
        if (map.exact) {
          valid[0] = map.window(item, len, first, width, chars, &p, &hlen);
        } else {
          WordSrc const at(bytes, mis + p);
          int32_t const here = base + static_cast<int32_t>(p);
          valid[0] = window_at(at, row + here, n - here + beyond, len - p, first && p == 0, all_ascii, width, &hlen);
        }
        WordSrc const src[1] = {WordSrc(bytes, mis + p)};
        if (valid[0]) hash(src, hlen, hv);
      }
      sink(valid, hv);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

}  // namespace nvtext_amd
