// The minimum of the 64-bit permutations ((h * a + b) mod 2^64) mod p, p = 2^61 - 1, over many hashes h, with the products
// computed to 16 bits by the matrix cores and only those of the few blocks of hashes that can hold the minimum computed exactly.
//
// What is minimised is, up to an addend of at most 7 (and the wrap from p to 0), the low 61 bits of h * a + b, that is the
// fraction X = frac((h * a + b) / 2^61).  With the hash cut into 2-bit digits u_i (i = 0 .. 30) X is the fraction of
//     b / 2^61 + sum over i of u_i * f_i,   f_i = frac(a * 4^i / 2^61),
// a matrix product of the digits of 32 hashes with the fractions of 32 parameters.  The f_i are rounded to the nearest
// multiple of 2^-16 (a unit) and cut into four pieces of 4, 5, 5 and 2 bits, which fp6 (e2m3) holds exactly, the digits are
// 2-bit patterns that fp4 (e2m1) reads as u / 2; a K-block of 32 elements of v_mfma_scale_f32_32x32x64_f8f6f4 takes the 31
// digits with one piece, whose weight is the block's scale.  Two instructions give 1,024 sums of all four
// pieces, exact in units: they start from 6.0, so that every sum lies in [4, 8), where an fp32 step is one unit, and the
// fraction is the low 16 bits of the pattern: 16-bit minima take the sums as they are.  Element 31 adds b and what the
// rounding may have taken away, so that the fraction found is always 1 to `slack` units above X, modulo 1: a product can
// only be less than v if its fraction is at most that of v plus the slack.
#pragma once

#include "common.cuh"

namespace nvtext_amd {
namespace filter64 {

using Sums = float __attribute__((ext_vector_type(16)));
using V8   = int __attribute__((ext_vector_type(8)));

constexpr int kGroup       = 32;             // parameters of one matrix instruction
constexpr int kUnits       = 16;             // bits of a fraction
constexpr int kUnitShift   = 61 - kUnits;    // a unit is 2^45 of a product
constexpr uint64_t kPrime  = (1ull << 61) - 1;
constexpr float kStart     = 6.0f;           // what the sums start from: its low 16 bits are zeros

// What the host side of a call lays out for a group of 32 parameters: the registers of the two matrix instructions, lane
// by lane, and the slack of every parameter.
struct alignas(16) Group {
  uint32_t pieces[2][6][kWave];  // 32 numbers of 6 bits a lane; lanes below 32: pieces 0 and 2, the others: 1 and 3
  uint32_t slack[kGroup];        // units
};

// The scale of a lane's pieces in the first and in the second instruction (as fp4 and fp6 read them, a product of a digit
// and a piece is worth 2^-4): a unit is 2^-21 of the sums, the pieces weigh 2^12, 2^7, 2^2 and 1 units.
__device__ __forceinline__ int scale_of(int instruction, int lane)
{
  int const high = lane < kGroup ? 12 : 7, low = lane < kGroup ? 2 : 0;
  return 127 + 4 - 21 + (instruction == 0 ? high : low);
}
constexpr int kScaleOne = 127;

// A number of at most 16 in size as fp6 (e2m3), in eighths.
__host__ __device__ inline uint32_t fp6_eighths(int v) { return v < 0 ? 32u | static_cast<uint32_t>(-v) : static_cast<uint32_t>(v); }

// Piece j of n, |n| <= 2^15 units.
__host__ __device__ inline int piece_of(int32_t n, int j)
{
  int const d3 = ((n + 2) & 3) - 2;
  n            = (n - d3) >> 2;
  int const d2 = ((n + 16) & 31) - 16;
  n            = (n - d2) >> 5;
  int const d1 = ((n + 16) & 31) - 16;
  n            = (n - d1) >> 5;
  return j == 0 ? n : j == 1 ? d1 : j == 2 ? d2 : d3;
}

// The order of the digits in a lane's registers: what digits_of() below finds with a mask and a shift.
__host__ __device__ inline int element_of_digit(int i)
{
  int const half = i >> 4, within = i & 15;
  return half * 16 + (within & 1) * 8 + (within >> 1);
}

// The numbers n_i of one parameter and its slack.  n(i, value) is called for the 31 digits, then for element 31.
template <typename Put>
__host__ __device__ inline uint32_t lay_out(uint64_t a, uint64_t b, Put&& put)
{
  uint64_t const half = 1ull << (kUnitShift - 1);
  uint64_t c = a & kPrime, low = 0, high = 0;  // how far the rounding can take a sum of the digits down and up, thirds of it
  int64_t below = 0, above = 0;                // the range of the sums, thirds of it
  for (int i = 0; i < 31; ++i) {
    int32_t n       = static_cast<int32_t>((c + half) >> kUnitShift);
    int64_t const e = (static_cast<int64_t>(n) << kUnitShift) - static_cast<int64_t>(c);
    if (e < 0) low += static_cast<uint64_t>(-e); else high += static_cast<uint64_t>(e);
    if (n > (1 << (kUnits - 1))) n -= 1 << kUnits;
    if (n < 0) below -= n; else above += n;
    put(element_of_digit(i), n);
    c = (c << 2) & kPrime;
  }
  // the largest loss rounded up, and a unit more, so that a value that wraps at p wraps here too; even, because element
  // 31 counts twice
  uint64_t const need = (((b & kPrime) + 3 * low) >> kUnitShift) + 2;
  int32_t bias        = static_cast<int32_t>((need + 1) & ((1u << kUnits) - 2));
  // the sums have 64 wholes of room on either side (2^22 units around 6.0) and take at most 31.2 (every digit of a / 2^61 to the base 4
  // is 1, or 2)
  if (above > below) bias -= 1 << kUnits;
  put(31, bias / 2);
  return static_cast<uint32_t>((3 * (low + high)) >> kUnitShift) + 4;
}

// ((h * a + b) mod 2^64) mod p (cpp/src/text/minhash.cu:350-351)
__host__ __device__ inline uint64_t exact(uint64_t h, uint64_t a, uint64_t b)
{
  uint64_t const x = h * a + b;
  uint64_t const y = (x & kPrime) + (x >> 61);
  return y >= kPrime ? y - kPrime : y;
}

// The digits of a hash as the matrix instruction reads them, element 31 set to 1.0 (which counts as a digit of 2).
__device__ __forceinline__ V8 digits_of(uint64_t h)
{
  uint32_t const lo = static_cast<uint32_t>(h), hi = static_cast<uint32_t>(h >> 32);
  V8 d              = {};
  d[0]              = static_cast<int>(lo & 0x33333333u);
  d[1]              = static_cast<int>((lo >> 2) & 0x33333333u);
  d[2]              = static_cast<int>(hi & 0x33333333u);
  d[3]              = static_cast<int>(((hi >> 2) & 0x03333333u) | 0x20000000u);
  return d;
}

__device__ __forceinline__ Sums sums_of(V8 const& digits, const uint32_t (&p0)[6], const uint32_t (&p1)[6], int scale0, int scale1, Sums const& start)
{
  V8 b0 = {}, b1 = {};
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    b0[k] = static_cast<int>(p0[k]);
    b1[k] = static_cast<int>(p1[k]);
  }
  constexpr int kFp4 = 4, kFp6 = 2;
  Sums const s = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(digits, b0, start, kFp4, kFp6, 0, kScaleOne, 0, scale0);
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(digits, b1, s, kFp4, kFp6, 0, kScaleOne, 0, scale1);
}

// The least fraction of a lane's sixteen sums, by two-way minima of 16 bits: they issue every two cycles (2.2 measured), a
// three-way one takes 8.9, and packed in pairs they need what packs them.  (The compiler forms the three-way ones, so only the
// first eight are its own: it also waits for the matrix cores there.)
__device__ __forceinline__ uint32_t least_of(Sums const& s)
{
  uint32_t k[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) k[r] = __builtin_elementwise_min(static_cast<uint16_t>(__float_as_uint(s[2 * r])), static_cast<uint16_t>(__float_as_uint(s[2 * r + 1])));
#pragma unroll
  for (int d = 4; d >= 1; d >>= 1)
#pragma unroll
    for (int r = 0; r < d; ++r) asm("v_min_u16 %0, %1, %2" : "=v"(k[r]) : "v"(k[r]), "v"(k[r + d]));
  return k[0];
}

// One wavefront lays a group out: lane l parameter l % 32.
__device__ __forceinline__ void prepare_group(const uint64_t* a, const uint64_t* b, int32_t P, int32_t group, Group* to, int lane)
{
  int32_t const j = min(group * kGroup + (lane & (kGroup - 1)), P - 1);
  int const first = lane < kGroup ? 0 : 1;
  uint32_t w[2][6] = {};
  uint32_t const slack = lay_out(a[j], b[j], [&](int element, int32_t n) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      uint32_t const v  = fp6_eighths(piece_of(n, first + 2 * k));
      uint32_t const at = 6u * static_cast<uint32_t>(element);
#pragma unroll
      for (uint32_t d = 0; d < 6; ++d) {  // (the registers are not indexed)
        uint32_t const shifted = at >= 32 * d ? (at - 32 * d < 32 ? v << (at - 32 * d) : 0u) : (32 * d - at < 6 ? v >> (32 * d - at) : 0u);
        w[k][d] |= shifted;
      }
    }
  });
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int d = 0; d < 6; ++d) to->pieces[k][d][lane] = w[k][d];
  if (lane < kGroup) to->slack[lane] = slack;
}

}  // namespace filter64
}  // namespace nvtext_amd
