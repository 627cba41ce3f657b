// Host check of the hashes in cudf_amd/csrc/murmur.cuh at lengths around their blocks and up to the largest a window can
// have, against the published algorithm with 64-bit places.  Key byte i is what Bytes says, so that no key is in memory;
// a read further back than the last ones, which a place that has wrapped makes, ends the program.
// (What the header takes from the compiler for the GPU is given here.)
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <algorithm>

static inline uint32_t alignbit(uint32_t hi, uint32_t lo, uint32_t n) { return static_cast<uint32_t>(((static_cast<uint64_t>(hi) << 32) | lo) >> (n & 31)); }
#define __builtin_amdgcn_alignbit alignbit
#include <hip/hip_runtime.h>
using std::max;
using std::min;
#include "murmur.cuh"

static inline uint32_t key_dword(uint64_t k) { return static_cast<uint32_t>(k) * 0x9E3779B1u ^ static_cast<uint32_t>(k >> 7); }
static inline uint64_t key_byte(uint64_t i) { return key_dword(i / 4) >> (8 * (i % 4)) & 0xFFu; }

template <bool IN_TILE>
struct Bytes {
  static constexpr bool kInTile = IN_TILE;
  mutable uint32_t furthest = 0;
  uint32_t byte(uint32_t i) const { return static_cast<uint32_t>(key_byte(i)); }
  uint32_t dword(uint32_t k) const
  {
    if (k + 8 < furthest) {
      std::printf("a read at dword %u after one at %u\n", k, furthest);
      std::exit(1);
    }
    furthest = std::max(furthest, k);
    return key_dword(k);
  }
};

static uint64_t rotl(uint64_t x, int r) { return (x << r) | (x >> (64 - r)); }
static uint64_t mix(uint64_t k)
{
  k = (k ^ (k >> 33)) * 0xff51afd7ed558ccdull;
  k = (k ^ (k >> 33)) * 0xc4ceb9fe1a85ec53ull;
  return k ^ (k >> 33);
}
static uint64_t published64(uint64_t len, uint64_t seed)
{
  uint64_t const c1 = 0x87c37b91114253d5ull, c2 = 0x4cf5ad432745937full;
  uint64_t h1 = seed, h2 = seed;
  for (uint64_t b = 0; b < len / 16; ++b) {
    uint64_t const k1 = key_dword(4 * b) | static_cast<uint64_t>(key_dword(4 * b + 1)) << 32, k2 = key_dword(4 * b + 2) | static_cast<uint64_t>(key_dword(4 * b + 3)) << 32;
    h1 = (rotl(h1 ^ rotl(k1 * c1, 31) * c2, 27) + h2) * 5 + 0x52dce729;
    h2 = (rotl(h2 ^ rotl(k2 * c2, 33) * c1, 31) + h1) * 5 + 0x38495ab5;
  }
  uint64_t k[2] = {0, 0};
  for (uint64_t i = len / 16 * 16; i < len; ++i) k[i % 16 / 8] |= key_byte(i) << (8 * (i % 8));
  h1 ^= rotl(k[0] * c1, 31) * c2 ^ len;
  h2 ^= rotl(k[1] * c2, 33) * c1 ^ len;
  h1 += h2;
  h2 += h1;
  return mix(h1) + mix(h2);
}
static uint32_t published32(uint64_t len, uint32_t seed)
{
  auto const rot   = [](uint32_t x, int r) { return (x << r) | (x >> (32 - r)); };
  auto const block = [&](uint32_t k) { return rot(k * 0xcc9e2d51u, 15) * 0x1b873593u; };
  uint32_t h = seed, rest = 0;
  for (uint64_t b = 0; b < len / 4; ++b) h = rot(h ^ block(key_dword(b)), 13) * 5 + 0xe6546b64u;
  for (uint64_t i = len / 4 * 4; i < len; ++i) rest |= static_cast<uint32_t>(key_byte(i)) << (8 * (i % 4));
  if (len % 4) h ^= block(rest);
  h ^= static_cast<uint32_t>(len);
  h = (h ^ (h >> 16)) * 0x85ebca6bu;
  h = (h ^ (h >> 13)) * 0xc2b2ae35u;
  return h ^ (h >> 16);
}

static void check(bool same, uint32_t len)
{
  if (same) return;
  std::printf("%u bytes: another hash\n", len);
  std::exit(1);
}
template <int N, bool IN_TILE>
static void check64(uint32_t len)
{
  Bytes<IN_TILE> const src[N] = {};
  uint64_t h[N];
  nvtext_amd::murmur3_x64_128_lo<N>(src, len, 7, h);
  for (uint64_t const v : h) check(v == published64(len, 7), len);
}
static void check32(uint32_t len)
{
  Bytes<false> const src[1] = {};
  uint32_t h[1];
  nvtext_amd::murmur3_x86_32<1>(src, len, 42, h);
  check(h[0] == published32(len, 42), len);
}

int main()
{
  for (uint32_t len = 0; len <= 100; ++len) {
    check64<2, true>(len);
    check64<1, false>(len);
    check32(len);
  }
  check64<1, false>(0xFFFFFFF1u);
  check64<1, false>(0xFFFFFFFFu);
  std::puts("ok");
}
