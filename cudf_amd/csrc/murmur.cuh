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

__device__ __forceinline__ uint32_t keep_low_bytes(uint32_t v, int nbytes)
{
  // nbytes in [0, 4]
  return nbytes >= 4 ? v : (v & ((1u << (8 * nbytes)) - 1u));
}

// Byte source over a dword array (an LDS tile): window byte i lives at byte offset base+i.
// dword(k), bytes 4k to 4k + 3 of the window, may read up to 11 bytes past the window (callers mask what they do not need).
// (A shift of two aligned dwords: an unaligned read of LDS takes a cycle a lane.)
struct WordSrc {
  static constexpr bool kInTile = true;  // its windows are no longer than a tile of a row
  const uint32_t* at;  // the dword with the window's first byte
  uint32_t mis;        // where in it
  __device__ __forceinline__ WordSrc(const uint32_t* w, uint32_t base) : at(w + (base >> 2)), mis(base & 3u) {}
  __device__ __forceinline__ uint32_t byte(uint32_t i) const { return reinterpret_cast<const uint8_t*>(at)[mis + i]; }
  __device__ __forceinline__ uint32_t dword(uint32_t k) const { return __builtin_amdgcn_alignbit(at[k + 1], at[k], 8u * mis); }
};

// Byte source over global memory that never touches a byte at or past `avail`
// (slow; used only for windows too wide for the LDS tile).
struct BoundedSrc {
  static constexpr bool kInTile = false;
  const uint8_t* p;
  int64_t avail;
  __device__ __forceinline__ uint32_t byte(uint32_t i) const { return p[i]; }
  __device__ __forceinline__ uint32_t dword(uint32_t k) const
  {
    uint32_t v = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (4 * static_cast<int64_t>(k) + j < avail) v |= static_cast<uint32_t>(p[4 * k + j]) << (8 * j);
    return v;
  }
};

// The hashes take N windows of one length at a time, step by step: their chains of reads and multiplications run side by side.

// Hashes of window bytes [0, len) of every `src` before their final mix.  The mix is a bijection that keeps 0, so where hashes
// are only compared with one another and with 0 these do as well.
template <int N, typename Src>
__device__ __forceinline__ void murmur3_x86_32_unmixed(Src const (&src)[N], uint32_t len, uint32_t seed, uint32_t (&h)[N])
{
  uint32_t const c1 = 0xcc9e2d51u, c2 = 0x1b873593u;
  uint32_t const blocks = len >> 2;
#pragma unroll
  for (int n = 0; n < N; ++n) h[n] = seed;
  for (uint32_t i = 0; i < blocks; ++i) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      uint32_t const k1 = rotl32(src[n].dword(i) * c1, 15) * c2;
      h[n]              = rotl32(h[n] ^ k1, 13) * 5u + 0xe6546b64u;
    }
  }
  uint32_t const rem = len & 3u;
  if (rem) {
#pragma unroll
    for (int n = 0; n < N; ++n) h[n] ^= rotl32(keep_low_bytes(src[n].dword(blocks), static_cast<int>(rem)) * c1, 15) * c2;
  }
#pragma unroll
  for (int n = 0; n < N; ++n) h[n] ^= len;
}

template <int N, typename Src>
__device__ __forceinline__ void murmur3_x86_32(Src const (&src)[N], uint32_t len, uint32_t seed, uint32_t (&h)[N])
{
  murmur3_x86_32_unmixed<N>(src, len, seed, h);
#pragma unroll
  for (int n = 0; n < N; ++n) {
    uint32_t h1 = h[n];
    h1 ^= h1 >> 16;
    h1 *= 0x85ebca6bu;
    h1 ^= h1 >> 13;
    h1 *= 0xc2b2ae35u;
    h[n] = h1 ^ (h1 >> 16);
  }
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

// The first n bytes (0 .. 8) of v.
__device__ __forceinline__ uint64_t low_bytes64(uint64_t v, uint32_t n) { return n == 0 ? 0 : v & (~0ull >> (64u - 8u * n)); }

// First 64-bit words of MurmurHash3_x64_128 with h1 = h2 = seed over window bytes [0, len).  What is left of the key after
// its blocks of 16 is treated as a block is up to where the halves are mixed: zeros in place of missing bytes change nothing,
// and lanes with keys either side of 16 bytes go one way (before, the ones waited while the others did their blocks).
template <int N, typename Src>
__device__ __forceinline__ void murmur3_x64_128_lo(Src const (&src)[N], uint32_t len, uint64_t seed, uint64_t (&h)[N])
{
  uint64_t const c1 = 0x87c37b91114253d5ull, c2 = 0x4cf5ad432745937full;
  uint64_t h1[N], h2[N];
#pragma unroll
  for (int n = 0; n < N; ++n) h1[n] = h2[n] = seed;
  // (behind the last block of a length just below 2^32 the place of the next one has wrapped: the byte before it tells)
  bool more = len != 0;
  for (uint32_t t = 0; more; t += 16, more = Src::kInTile ? t < len : t - 1u < len - 1u) {
    uint32_t const left = len - t, at = t / 4u;
#pragma unroll
    for (int n = 0; n < N; ++n) {
      uint64_t const k1 = static_cast<uint64_t>(src[n].dword(at + 1)) << 32 | src[n].dword(at);
      h1[n] ^= rotl64(low_bytes64(k1, min(left, 8u)) * c1, 31) * c2;
    }
    uint64_t k2[N];
#pragma unroll
    for (int n = 0; n < N; ++n) k2[n] = 0;
    if (left > 8) {
#pragma unroll
      for (int n = 0; n < N; ++n) {
        uint64_t const k = static_cast<uint64_t>(src[n].dword(at + 3)) << 32 | src[n].dword(at + 2);
        k2[n]            = rotl64(low_bytes64(k, min(left, 16u) - 8u) * c2, 33) * c1;
      }
    }
    if (left >= 16) {
#pragma unroll
      for (int n = 0; n < N; ++n) {
        h1[n] = (rotl64(h1[n], 27) + h2[n]) * 5 + 0x52dce729;
        h2[n] = (rotl64(h2[n] ^ k2[n], 31) + h1[n]) * 5 + 0x38495ab5;
      }
    } else {
#pragma unroll
      for (int n = 0; n < N; ++n) h2[n] ^= k2[n];
    }
  }
#pragma unroll
  for (int n = 0; n < N; ++n) {
    h1[n] ^= len;
    h2[n] ^= len;
    h1[n] += h2[n];
    h2[n] += h1[n];
    h[n] = fmix64(h1[n]) + fmix64(h2[n]);
  }
}

}  // namespace nvtext_amd
