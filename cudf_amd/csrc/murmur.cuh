// MurmurHash3_x86_32 and MurmurHash3_x64_128 (word 0) over a byte range that sits in a
// dword array (LDS tile or global memory), read as unaligned little-endian dwords.
// The arithmetic is the published MurmurHash3 the reference reaches through
// cuco::murmurhash3_32 / cuco::murmurhash3_x64_128
// (cpp/include/cudf/hashing/detail/murmurhash3_x86_32.cuh:21-46,
//  cpp/include/cudf/hashing/detail/murmurhash3_x64_128.cuh:18-43).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nvtext_amd {

__device__ __forceinline__ uint32_t rotl32(uint32_t x, int r) { return __builtin_amdgcn_alignbit(x, x, 32 - r); }
__device__ __forceinline__ uint64_t rotl64(uint64_t x, int r) { return (x << r) | (x >> (64 - r)); }

// Dword starting at byte offset `o` of the dword array `w` (reads w[o/4] and w[o/4+1]).
__device__ __forceinline__ uint32_t load_u32_at(const uint32_t* w, uint32_t o)
{
  uint32_t const i  = o >> 2;
  uint32_t const lo = w[i];
  uint32_t const hi = w[i + 1];
  return __builtin_amdgcn_alignbit(hi, lo, (o & 3u) * 8u);
}

__device__ __forceinline__ uint32_t keep_low_bytes(uint32_t v, int nbytes)
{
  // nbytes in [0, 4]
  return nbytes >= 4 ? v : (v & ((1u << (8 * nbytes)) - 1u));
}

// Byte source over a dword array (an LDS tile): window byte i lives at byte offset base+i.
// u32(i) may read up to 11 bytes past the window (callers mask what they do not need).
struct WordSrc {
  const uint32_t* w;
  uint32_t base;
  __device__ __forceinline__ uint32_t byte(uint32_t i) const { return reinterpret_cast<const uint8_t*>(w)[base + i]; }
  __device__ __forceinline__ uint32_t u32(uint32_t i) const { return load_u32_at(w, base + i); }
};

// Byte source over global memory that never touches a byte at or past `avail`
// (slow; used only for windows too wide for the LDS tile).
struct BoundedSrc {
  const uint8_t* p;
  int64_t avail;
  __device__ __forceinline__ uint32_t byte(uint32_t i) const { return p[i]; }
  __device__ __forceinline__ uint32_t u32(uint32_t i) const
  {
    uint32_t v = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (static_cast<int64_t>(i) + k < avail) v |= static_cast<uint32_t>(p[i + k]) << (8 * k);
    return v;
  }
};

// Hash of window bytes [0, len) of `src` before its final mix.  The mix is a bijection that keeps 0, so where hashes are
// only compared with one another and with 0 this does as well.
template <typename Src>
__device__ __forceinline__ uint32_t murmur3_x86_32_unmixed(Src const& src, uint32_t len, uint32_t seed)
{
  uint32_t const c1 = 0xcc9e2d51u, c2 = 0x1b873593u;
  uint32_t h1           = seed;
  uint32_t const blocks = len >> 2;
  for (uint32_t i = 0; i < blocks; ++i) {
    uint32_t k1 = src.u32(4 * i);
    k1 *= c1;
    k1 = rotl32(k1, 15);
    k1 *= c2;
    h1 ^= k1;
    h1 = rotl32(h1, 13);
    h1 = h1 * 5u + 0xe6546b64u;
  }
  uint32_t const rem = len & 3u;
  if (rem) {
    uint32_t k1 = keep_low_bytes(src.u32(4 * blocks), static_cast<int>(rem));
    k1 *= c1;
    k1 = rotl32(k1, 15);
    k1 *= c2;
    h1 ^= k1;
  }
  return h1 ^ len;
}

template <typename Src>
__device__ __forceinline__ uint32_t murmur3_x86_32(Src const& src, uint32_t len, uint32_t seed)
{
  uint32_t h1 = murmur3_x86_32_unmixed(src, len, seed);
  h1 ^= h1 >> 16;
  h1 *= 0x85ebca6bu;
  h1 ^= h1 >> 13;
  h1 *= 0xc2b2ae35u;
  h1 ^= h1 >> 16;
  return h1;
}

__device__ __forceinline__ uint64_t fmix64(uint64_t k)
{
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  k *= 0xc4ceb9fe1a85ec53ull;
  k ^= k >> 33;
  return k;
}

template <typename Src>
__device__ __forceinline__ uint64_t load_u64(Src const& src, uint32_t i)
{
  return (static_cast<uint64_t>(src.u32(i + 4)) << 32) | src.u32(i);
}

// The first n bytes (0 .. 8) of v.
__device__ __forceinline__ uint64_t low_bytes64(uint64_t v, uint32_t n) { return n == 0 ? 0 : v & (~0ull >> (64u - 8u * n)); }

// First 64-bit word of MurmurHash3_x64_128 with h1 = h2 = seed over window bytes [0, len).  What is left of the key after
// its blocks of 16 is treated as a block is up to where the halves are mixed: zeros in place of missing bytes change nothing,
// and lanes with keys either side of 16 bytes go one way (before, the ones waited while the others did their blocks).
template <typename Src>
__device__ __forceinline__ uint64_t murmur3_x64_128_lo(Src const& src, uint32_t len, uint64_t seed)
{
  uint64_t const c1 = 0x87c37b91114253d5ull, c2 = 0x4cf5ad432745937full;
  uint64_t h1 = seed, h2 = seed;
  for (uint32_t t = 0; t < len; t += 16) {
    uint32_t const left = len - t;
    uint64_t k1 = low_bytes64(load_u64(src, t), min(left, 8u));
    k1 *= c1;
    k1 = rotl64(k1, 31);
    k1 *= c2;
    h1 ^= k1;
    uint64_t k2 = 0;
    if (left > 8) {
      k2 = low_bytes64(load_u64(src, t + 8), min(left, 16u) - 8u);
      k2 *= c2;
      k2 = rotl64(k2, 33);
      k2 *= c1;
    }
    if (left >= 16) {
      h1 = rotl64(h1, 27);
      h1 += h2;
      h1 = h1 * 5 + 0x52dce729;
      h2 ^= k2;
      h2 = rotl64(h2, 31);
      h2 += h1;
      h2 = h2 * 5 + 0x38495ab5;
    } else {
      h2 ^= k2;
    }
  }
  h1 ^= len;
  h2 ^= len;
  h1 += h2;
  h2 += h1;
  h1 = fmix64(h1);
  h2 = fmix64(h2);
  h1 += h2;
  return h1;
}

}  // namespace nvtext_amd
