// minhash / minhash64 for gfx950.
//
// Replaces the reference's three-kernel pipeline (cpp/src/text/minhash.cu:87-157 seed
// hashes into a chars-sized temporary, 281-376 permutation kernel re-reading it,
// 390-424 size partitioning) with one fused pass and no chars-sized temporary:
//
//   * a wavefront owns a section of a row.  Per 256-position tile it stages the bytes
//     in LDS (coalesced aligned 16-byte loads), hashes the windows with lanes <-> window
//     starts, and compacts the hashes into LDS;
//   * it then switches to lanes <-> parameters.  32-bit hashes: every lane keeps K (a, b) pairs and
//     K running minima in registers and streams the tile's hashes through LDS
//     broadcast reads, so the inner loop is v_mad_u64_u32 + v_min only (MinimaAll).  64-bit hashes:
//     the matrix cores find which few of them can give the minimum, and only their products are
//     computed (Minima64, filter64.cuh);
//   * a wavefront does a row alone, or a part of it: rows are cut into even parts of at most 4.2 KB
//     (64-bit hashes: 6 KiB; of fewer bytes in a column too small to give every wavefront of the device
//     several of that size), the parts of a row meet in the result with an atomic minimum, and the
//     wavefronts take short parts several at a time;
//   * in a tile with characters of more than one byte the wavefront lists the characters first,
//     so that a lane takes a character and reads its window's length instead of walking to it;
//     hashes that the wavefront has folded lately are dropped (a minimum does not mind).
//
// Null rows get no output slot (the reference drops them with purge_nonempty_nulls,
// minhash.cu:626-628), empty rows are all zeros (minhash.cu:318).
#include "common.cuh"
#include "filter64.cuh"
#include "murmur.cuh"
#include "windows.cuh"

#include <algorithm>
#include <limits>
#include <mutex>
#include <type_traits>

// Scratch of nvtext_amd_minhash_preallocated, the entry point that allocates nothing: the part counts of the
// rows (rows + 1 values) and behind them the sums of the plan and the counters of the units of work.  Every device holds
// its own copy of the array for as long as the library is loaded (4.2 MB).
constexpr int32_t kPreallocatedMaxRows = NVTEXT_AMD_MINHASH_PREALLOCATED_MAX_ROWS;
constexpr size_t kScratchPrefixBytes   = (static_cast<size_t>(kPreallocatedMaxRows) + 1 + 63) / 64 * 64 * sizeof(uint32_t);
constexpr int kSumTiles                = 1024;  // tiles of rows at most, whose sums the plan of a larger column adds up
constexpr int kCounterGroups           = 32;    // counters of units of work
constexpr int kCounterLine             = 16;    // 64-bit words from one to the next: a 128-byte line each
constexpr size_t kPlanBytes            = ((kCounterGroups + 1) * kCounterLine + kSumTiles) * sizeof(uint64_t);
static __device__ __align__(256) unsigned char scratch[kScratchPrefixBytes + kPlanBytes];

namespace nvtext_amd {
namespace {

template <typename T>
struct HashTraits;
template <>
struct HashTraits<uint32_t> {
  // (0 is no hash: minhash.cu:141, 237)
  template <int N, typename Src>
  static __device__ __forceinline__ void hash(Src const (&src)[N], uint32_t len, uint32_t seed, uint32_t (&h)[N])
  {
    murmur3_x86_32<N>(src, len, seed, h);
#pragma unroll
    for (int n = 0; n < N; ++n) h[n] = max(h[n], 1u);
  }
  // Permutation (minhash.cu:350-351) in uint32 arithmetic: the product and sum wrap mod 2^32, after
  // which "% (2^61-1)" and "& max" change nothing: (hv * a + b), see Fold.
};
template <>
struct HashTraits<uint64_t> {
  template <int N, typename Src>
  static __device__ __forceinline__ void hash(Src const (&src)[N], uint32_t len, uint64_t seed, uint64_t (&h)[N])
  {
    murmur3_x64_128_lo<N>(src, len, seed, h);  // minhash.cu:138: first word of the 128-bit hash
#pragma unroll
    for (int n = 0; n < N; ++n) h[n] += h[n] == 0 ? 1u : 0u;
  }
  // Permutation (minhash.cu:350-351): ((hv*a + b) mod 2^64) % (2^61-1), see filter64.cuh.
};

// How the lanes of a wavefront share the work when there are at most 32 parameters: `groups` sets of `ppad` lanes
// (both powers of two, groups <= 16), lane l holding parameter l % ppad and folding the trips l / ppad,
// l / ppad + groups, ...  The sets are combined with a butterfly of minima before the results leave the registers.
struct Packing {
  int32_t ppad;    // lanes per set; 64 when every lane has its own parameter
  int32_t groups;  // sets per wavefront
  __device__ __forceinline__ int param_lane(int lane) const { return lane & (ppad - 1); }
  __device__ __forceinline__ uint32_t first(int lane, uint32_t per_trip) const { return static_cast<uint32_t>(lane / ppad) * per_trip; }
  __device__ __forceinline__ uint32_t stride(uint32_t per_trip) const { return static_cast<uint32_t>(groups) * per_trip; }
  template <typename T>
  __device__ __forceinline__ T combine(T m) const
  {
    for (int d = ppad; d < kWave; d <<= 1) {
      T const other = __shfl_xor(m, d);
      m             = min(m, other);
    }
    return m;
  }
};

__host__ __device__ inline Packing packing_for(int32_t P)
{
  if (P > 32) return Packing{kWave, 1};
  int32_t ppad = 4;  // at most 16 sets, so that the padding of a tile's hashes fits one wavefront-wide store
  while (ppad < P) ppad <<= 1;
  return Packing{ppad, kWave / ppad};
}

// Folds the compacted hashes first, first + 1, .. of every `stride` (the count padded to a multiple of the stride)
// into m[K]; lanes <-> parameters.  A wavefront whose lanes all hold different parameters folds every hash
// (first 0, stride = the hashes of one trip); with few parameters the lanes form groups that hold the same
// parameters and fold every other trip each (see Packing).
constexpr uint32_t kFoldTrip = 4;
template <int K>
__device__ __forceinline__ void fold_all(const uint32_t* hashes, uint32_t padded, uint32_t first, uint32_t stride, const uint32_t (&a)[K],
                                       const uint32_t (&b)[K], uint32_t (&m)[K])
{
  for (uint32_t i = first; i < padded; i += stride) {
    uint32_t const h0 = hashes[i], h1 = hashes[i + 1], h2 = hashes[i + 2], h3 = hashes[i + 3];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      // one v_mad_u64_u32 per product, one v_min3_u32 per two products
      uint32_t const r0 = h0 * a[k] + b[k];
      uint32_t const r1 = h1 * a[k] + b[k];
      uint32_t const r2 = h2 * a[k] + b[k];
      uint32_t const r3 = h3 * a[k] + b[k];
      m[k]              = min(min(m[k], r0), r1);
      m[k]              = min(min(m[k], r2), r3);
    }
  }
}

// The same for 64-bit hashes, every product computed whole (see filter64.cuh for the permutation).
//
// ((h * a + b) mod 2^64) folded once mod 2^61 - 1, that is (x & p) + (x >> 61) for the 64-bit x, at most p + 7, for two
// hashes and one (a, b): x = h.lo * a.lo + b is a 64-bit multiply-add; the two cross products, of which only the low
// dwords count, are two more, chained, and their sum goes to the high dword of x with a 32-bit add; the fold is a shift
// and a mask of that dword and one more multiply-add (q * 1 + x) for the carry.  The chained pairs of the two hashes stand
// interleaved, so that neither waits for its own first half.
__device__ __forceinline__ void fold_pair(uint64_t h0, uint64_t h1, uint64_t a, uint64_t b, uint32_t one, uint64_t* y0, uint64_t* y1)
{
  uint32_t const al = static_cast<uint32_t>(a), ah = static_cast<uint32_t>(a >> 32);
  uint32_t const l0 = static_cast<uint32_t>(h0), u0 = static_cast<uint32_t>(h0 >> 32);
  uint32_t const l1 = static_cast<uint32_t>(h1), u1 = static_cast<uint32_t>(h1 >> 32);
  uint64_t c0, c1;
  asm("v_mad_u64_u32 %0, vcc, %2, %6, 0\n\t"
      "v_mad_u64_u32 %1, vcc, %4, %6, 0\n\t"
      "v_mad_u64_u32 %0, vcc, %3, %7, %0\n\t"
      "v_mad_u64_u32 %1, vcc, %5, %7, %1"
      : "=&v"(c0), "=&v"(c1)
      : "v"(l0), "v"(u0), "v"(l1), "v"(u1), "v"(ah), "v"(al)
      : "vcc");
  uint64_t const x0 = static_cast<uint64_t>(l0) * al + b;
  uint64_t const x1 = static_cast<uint64_t>(l1) * al + b;
  uint32_t xh0      = static_cast<uint32_t>(x0 >> 32) + static_cast<uint32_t>(c0);
  uint32_t xh1      = static_cast<uint32_t>(x1 >> 32) + static_cast<uint32_t>(c1);
  uint32_t const q0 = xh0 >> 29, q1 = xh1 >> 29;
  xh0 &= 0x1FFFFFFFu;
  xh1 &= 0x1FFFFFFFu;
  *y0 = static_cast<uint64_t>(q0) * one + ((static_cast<uint64_t>(xh0) << 32) | static_cast<uint32_t>(x0));
  *y1 = static_cast<uint64_t>(q1) * one + ((static_cast<uint64_t>(xh1) << 32) | static_cast<uint32_t>(x1));
}

// min of two values below 2^62 in one instruction: such bit patterns are non-negative finite doubles (or denormals, which
// this code object keeps: float_denorm_mode_16_64 = 3), and those order like the integers.  An operand that is all ones
// (the start value, a NaN pattern) loses to the other.
__device__ __forceinline__ uint64_t min_below_2_62(uint64_t m, uint64_t y)
{
  uint64_t r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(m), "v"(y));
  return r;
}

// The least of such values over the lanes.  (By moves of the lanes' registers: exchanged through LDS, two reads a step one after
// the other, it was what a short part waited for longest: 1400 rows of 300 bytes, 256 parameters 56 -> 46 us.)
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint64_t min_with_lane(uint64_t v)
{
  uint32_t const lo = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(-1, static_cast<int>(v), CTRL, ROW_MASK, 0xF, false));
  uint32_t const hi = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(-1, static_cast<int>(v >> 32), CTRL, ROW_MASK, 0xF, false));
  return min_below_2_62(v, (static_cast<uint64_t>(hi) << 32) | lo);
}
__device__ __forceinline__ uint64_t least_of_lanes(uint64_t v)
{
  v = min_with_lane<0x111, 0xF>(v);  // row_shr:1, :2, :4, :8
  v = min_with_lane<0x112, 0xF>(v);
  v = min_with_lane<0x114, 0xF>(v);
  v = min_with_lane<0x118, 0xF>(v);
  v = min_with_lane<0x142, 0xA>(v);  // row_bcast:15, :31
  v = min_with_lane<0x143, 0xC>(v);
  return wave_bcast64(v, kWave - 1);
}

template <int K>
__device__ __forceinline__ void fold_all(const uint64_t* hashes, uint32_t padded, uint32_t first, uint32_t stride, const uint64_t (&a)[K],
                                         const uint64_t (&b)[K], uint64_t (&m)[K])
{
  // The last "subtract p if y >= p" is left out: it takes a y whose top dword is at least 0x1FFFFFFF (one product in
  // 2^29), which a running maximum tells; if there is one all hashes are folded again exactly.  (Values that ought to
  // have been reduced are above all that are, so that they have displaced none.)
  uint32_t top = 0;
  uint32_t one;  // the number 1 where the compiler does not see it: q * one + x stays one multiply-add
  asm("s_mov_b32 %0, 1" : "=s"(one));
  for (uint32_t i = first; i < padded; i += stride) {
    uint64_t h[kFoldTrip];
#pragma unroll
    for (uint32_t j = 0; j < kFoldTrip; ++j) h[j] = hashes[i + j];
#pragma unroll
    for (int k = 0; k < K; ++k) {
#pragma unroll
      for (uint32_t j = 0; j < kFoldTrip; j += 2) {
        uint64_t y0, y1;
        fold_pair(h[j], h[j + 1], a[k], b[k], one, &y0, &y1);
        top  = max(max(top, static_cast<uint32_t>(y0 >> 32)), static_cast<uint32_t>(y1 >> 32));
        m[k] = min_below_2_62(min_below_2_62(m[k], y0), y1);
      }
    }
  }
  if (ballot64(top >= 0x1FFFFFFFu) != 0) {
    // (every lane folds every hash here: a minimum does not mind the hashes of the other sets)
    for (uint32_t i = 0; i < padded; ++i) {
      uint64_t const h = hashes[i];
#pragma unroll
      for (int k = 0; k < K; ++k) m[k] = min(m[k], filter64::exact(h, a[k], b[k]));
    }
  }
}

// What the kernels are given of the parameters.
template <typename T>
struct Params {
  const T* a;
  const T* b;
  int32_t count;
  const filter64::Group* groups;  // 64-bit hashes only: the same, laid out for the matrix cores
};

// The minima of a row (or of a part of one) over the parameters of a chunk, by one wavefront: load() the chunk, reset(),
// fold() hashes out of LDS as often as needed (the number returned are left for the next time, in front, unless it is the
// last), finish(), each(put) calls put(j, minimum) for the parameters.

// Every product computed: K sets of 64 parameters, a lane has one of each set; with TAIL the parameters beyond the last full set, when
// there are at most 32 of them, are one more (a, b) pair per lane, shared out over sets of lanes as Packing describes, so
// that they cost the fold a share of a full set (4 parameters beyond 256: a sixteenth) instead of a whole one.
template <typename T_, int K, bool TAIL>
struct MinimaAll {
  using T = T_;
  struct Lds {};
  static constexpr int kParams = K * kWave;                       // of a chunk
  static constexpr int kSlots  = (K + (TAIL ? 1 : 0)) * kWave;    // (with TAIL there is one chunk)
  // wavefronts per SIMD that the registers are held to (64-bit hashes, 256 parameters: five spill nine registers, and
  // 20,000 lists of 200 elements take 306 us, with four 318)
  static constexpr int kSimdWaves = sizeof(T) == 4 ? 7 : 5;
  T a[K], b[K], m[K];
  T tail_a[1], tail_b[1], tail_m[1];
  Packing pk, tail_pk;
  int lane;

  static constexpr bool kCutUp = false;  // whether a chunk may have fewer parameters than it has room for (see minhash_parts_kernel)
  __device__ __forceinline__ MinimaAll(Lds*, int lane_, int32_t) : lane(lane_) {}
  __device__ __forceinline__ int32_t stride() const { return kParams; }
  __device__ __forceinline__ int32_t slots() const { return kSlots; }
  __device__ __forceinline__ void load(Params<T> const& p, int32_t chunk)
  {
    pk = K == 1 ? packing_for(p.count) : Packing{kWave, 1};
#pragma unroll
    for (int k = 0; k < K; ++k) {
      int32_t const j = chunk * kParams + pk.param_lane(lane) + kWave * k;
      a[k]            = j < p.count ? p.a[j] : T{0};
      b[k]            = j < p.count ? p.b[j] : T{0};
    }
    if (TAIL) {
      tail_pk         = packing_for(p.count - kParams);
      int32_t const j = kParams + tail_pk.param_lane(lane);
      tail_a[0]       = j < p.count ? p.a[j] : T{0};
      tail_b[0]       = j < p.count ? p.b[j] : T{0};
    }
  }
  __device__ __forceinline__ void reset()
  {
#pragma unroll
    for (int k = 0; k < K; ++k) m[k] = std::numeric_limits<T>::max();
    tail_m[0] = std::numeric_limits<T>::max();
  }
  // hashes: `count` of them, and room for 63 more
  __device__ __forceinline__ uint32_t fold(T* hashes, uint32_t count, bool)
  {
    wave_lds_fence();
    if (count == 0) return 0;
    // a duplicate never changes a minimum
    uint32_t stride = K > 1 ? kFoldTrip : pk.stride(kFoldTrip);  // a power of two, at most 64
    if (TAIL) stride = max(stride, tail_pk.stride(kFoldTrip));
    uint32_t const padded = (count + stride - 1u) & ~(stride - 1u);
    if (lane < static_cast<int>(padded - count)) hashes[count + lane] = hashes[0];
    wave_lds_fence();
    // the usual case keeps the loop counter out of the vector registers
    if (K > 1 || pk.groups == 1)
      fold_all<K>(hashes, padded, 0u, kFoldTrip, a, b, m);
    else
      fold_all<K>(hashes, padded, pk.first(lane, kFoldTrip), pk.stride(kFoldTrip), a, b, m);
    if (TAIL) fold_all<1>(hashes, padded, tail_pk.first(lane, kFoldTrip), tail_pk.stride(kFoldTrip), tail_a, tail_b, tail_m);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return 0;
  }
  __device__ __forceinline__ void finish()
  {
    if (K == 1) m[0] = pk.combine(m[0]);
    if (TAIL) tail_m[0] = tail_pk.combine(tail_m[0]);  // every set of lanes then holds the minima
  }
  template <typename Put>
  __device__ __forceinline__ void each(Put const& put) const
  {
    // (with fewer than 64 parameters the first lanes hold one each, in order)
#pragma unroll
    for (int k = 0; k < K; ++k) put(lane + kWave * k, m[k]);
    if (TAIL) put(kParams + lane, tail_m[0]);
  }
};

// 64-bit hashes: GROUPS groups of 32 parameters, AT_ONCE at a time, each product to 16 bits by the matrix cores (see filter64.cuh),
// 32 hashes at a time.  A lane has a parameter of every group and half of the hashes.  The hashes gather in LDS until kFoldFrom
// are there or the part ends; then, for every block of 32, the least of the lane's sixteen fractions is ranked, with the
// number of its half block below it, among the least three so far.  When all blocks are through, a lane takes one of the
// parameters of two groups, and the sixteen products of the half block that comes first are computed exactly; their minimum
// says which fractions can belong to a smaller one: the half block that comes second is computed as well if it is one of those,
// all hashes are if the third is (random parameters, counted over 40 sets of random hashes: of 256 hashes the second for 8 parameters
// in a hundred and the third for 0.3, of 450 14 and 1, of 670 19 and 1.5, of 1000 27 and 4).
// What bounds it: 1,024 products take 150 to 165 cycles of a SIMD, 86 of them the two matrix instructions, beside which the
// vector ALUs stand still but for some 20, 33 the sixteen-bit minima, 20 the ranking (with the shifts and three-way minima of
// whole dwords that put every single product in order before: 160 beside the matrix instructions; 20,011 long rows, 128
// parameters 3.73 -> 2.72 ms, 30,000 rows of 3000 bytes, 260 parameters 3.00 -> 2.06, 20,000 lists of 480 words, 256 parameters 627 -> 346 us).
template <int GROUPS, int AT_ONCE>
struct Minima64 {
  using T = uint64_t;
  static constexpr int kParams    = GROUPS * filter64::kGroup;
  static constexpr int kSlots     = kParams;
  static constexpr int kSimdWaves = AT_ONCE <= 2 ? 4 : 3;  // (the registers of 127 to 157 numbers)
  struct Lds {
    alignas(16) T minima[kParams];
  };
  Params<T> params;
  int32_t base;    // first parameter of the chunk
  int32_t groups;  // of the chunk: GROUPS, or fewer in a column with too few units of work for all wavefronts
  uint32_t warm;   // (see load)
  Lds* lds;
  int lane;
  static constexpr int kLeast  = GROUPS < 2 ? GROUPS : 2;  // groups that a chunk has at least
  static constexpr bool kCutUp = GROUPS > kLeast;

  // (with one group or two their number is known when this is compiled: 400,000 rows of several scripts, 64 parameters 2022 -> 2006 us)
  __device__ __forceinline__ Minima64(Lds* lds_, int lane_, int32_t groups_) : groups(kCutUp && groups_ != 0 ? groups_ : GROUPS), warm(0), lds(lds_), lane(lane_) {}
  __device__ __forceinline__ int32_t stride() const { return slots(); }  // parameters from a chunk to the next
  __device__ __forceinline__ int32_t slots() const { return groups * filter64::kGroup; }
  // What the first groups have in memory is asked for here, a cache line a lane, and waited for where it is used: the plan has
  // just written it, and a read then takes two microseconds.
  __device__ __forceinline__ void load(Params<T> const& p, int32_t chunk)
  {
    params = p;
    base   = chunk * slots();
    int32_t const first   = base / filter64::kGroup, last = (params.count - 1) / filter64::kGroup;
    const uint8_t* const at = reinterpret_cast<const uint8_t*>(params.groups + min(first, last));
    int32_t const size      = static_cast<int32_t>(sizeof(filter64::Group)) * min(kLeast, last - min(first, last) + 1);
    warm = *reinterpret_cast<const uint32_t*>(at + min(128 * lane, size - 4));
  }
  __device__ __forceinline__ void reset()
  {
    for (int j = lane; j < kParams; j += kWave) lds->minima[j] = std::numeric_limits<T>::max();
  }

  // The least product of the sixteen hashes of a half block.
  static __device__ __forceinline__ T exact(const T* hashes, uint32_t half_block, T a, T b)
  {
    // (hashes 4 .. 7, 12 .. 15, .. of a block for the upper half)
    const ulonglong2* const from = reinterpret_cast<const ulonglong2*>(hashes + (half_block >> 1) * 32u + (half_block & 1u) * 4u);
    T m          = std::numeric_limits<T>::max();
    uint32_t top = 0, one;
    asm("s_mov_b32 %0, 1" : "=s"(one));
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      ulonglong2 const h = from[(i >> 1) * 4 + (i & 1)];
      T y0, y1;
      fold_pair(h.x, h.y, a, b, one, &y0, &y1);
      top = max(max(top, static_cast<uint32_t>(y0 >> 32)), static_cast<uint32_t>(y1 >> 32));
      m   = min_below_2_62(min_below_2_62(m, y0), y1);
    }
    // (see fold_all: p and what is above it ought to have been reduced)
    if (ballot64(top >= 0x1FFFFFFFu) != 0) {
#pragma unroll 1
      for (int i = 0; i < 8; ++i) {
        ulonglong2 const h = from[(i >> 1) * 4 + (i & 1)];
        m = min(min(m, filter64::exact(h.x, a, b)), filter64::exact(h.y, a, b));
      }
    }
    return m;
  }

  // What no fraction of a product less than v exceeds.
  static __device__ __forceinline__ uint32_t limit_of(T v, uint32_t slack)
  {
    return static_cast<uint32_t>(min((v >> filter64::kUnitShift) + slack, static_cast<T>(0xFFFFu)));
  }

  struct Ranked {
    uint32_t first, second, third;
    // (what comes before stays in order: the old ones are read before they are written)
    __device__ __forceinline__ void add(uint32_t key)
    {
      third  = median(second, third, key);
      second = median(first, second, key);
      first  = min(first, key);
    }
    // The first three of both halves of the wavefront.
    __device__ __forceinline__ void merge_halves()
    {
      auto const f = __builtin_amdgcn_permlane32_swap(first, first, false, false);
      auto const s = __builtin_amdgcn_permlane32_swap(second, second, false, false);
      auto const t = __builtin_amdgcn_permlane32_swap(third, third, false, false);
      first  = min(f[0], f[1]);
      second = min(min(max(f[0], f[1]), s[0]), s[1]);
      third  = min(min(t[0], t[1]), min(max(f[0], s[1]), max(f[1], s[0])));
    }
  };

  // The parameters of two groups, a lane each (index j of the chunk; a single group: both halves have the same, the lower one
  // acts).  Lanes beyond the last parameter have its products, but go through nothing more for them: a row for which the last
  // of 260 parameters needs a second half block kept a wavefront busy with it 28 times over (100 rows of 2000 bytes 67 -> 33 us).
  __device__ __forceinline__ void settle(Ranked const& of_lower, Ranked const& of_upper, int j, bool two, const T* hashes, uint32_t count)
  {
    bool const upper = lane >= filter64::kGroup;
    bool const acts  = base + j < params.count && (two || !upper);
    Ranked const r{upper ? of_upper.first : of_lower.first, upper ? of_upper.second : of_lower.second, upper ? of_upper.third : of_lower.third};
    int32_t const at     = min(base + j, params.count - 1);
    T const a = params.a[at], b = params.b[at];
    uint32_t const slack = params.groups[at / filter64::kGroup].slack[at % filter64::kGroup];
    T m                  = min(lds->minima[j], exact(hashes, r.first & 0xFFFFu, a, b));
    uint64_t todo        = ballot64(acts && r.second >> 16 <= limit_of(m, slack));
    if (todo != 0) {
      // few parameters: the products of four of them at a time, sixteen lanes each
      if (acts) lds->minima[j] = m;
      wave_lds_fence();
      do {
        int who[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          who[i] = todo != 0 ? static_cast<int>(__builtin_ctzll(todo)) : who[i == 0 ? 0 : i - 1];
          todo &= todo - 1;
        }
        int const of          = lane < 32 ? (lane < 16 ? who[0] : who[1]) : (lane < 48 ? who[2] : who[3]);
        T const wa            = __shfl(static_cast<unsigned long long>(a), of), wb = __shfl(static_cast<unsigned long long>(b), of);
        uint32_t const half   = __shfl(r.second, of) & 0xFFFFu;
        uint32_t const within = static_cast<uint32_t>(lane) & 15u;
        T const v             = filter64::exact(hashes[(half >> 1) * 32u + (half & 1u) * 4u + (within >> 2) * 8u + (within & 3u)], wa, wb);
        unsigned long long* const to = reinterpret_cast<unsigned long long*>(&lds->minima[__shfl(j, of)]);
        if (v < *to) atomicMin(to, static_cast<unsigned long long>(v));
      } while (todo != 0);
      wave_lds_fence();
      m = lds->minima[j];
      for (todo = ballot64(acts && r.third >> 16 <= limit_of(m, slack)); todo != 0; todo &= todo - 1) {
        int const who = static_cast<int>(__builtin_ctzll(todo));
        T const wa = wave_bcast64(a, who), wb = wave_bcast64(b, who);
        T v = std::numeric_limits<T>::max();
        for (uint32_t i = lane; i < count; i += kWave) v = min(v, filter64::exact(hashes[i], wa, wb));
        v = least_of_lanes(v);
        if (lane == who) m = min(m, v);
      }
    }
    if (acts) lds->minima[j] = m;
  }

  template <int G>
  __device__ __forceinline__ void fold_groups(int32_t first, const T* hashes, uint32_t count)
  {
    asm("" : "+s"(first));  // (the pieces are read anew for every fold: not kept in registers while windows are hashed)
    asm volatile("" : : "v"(warm));
    // (the parameters are asked for before the blocks, so that they are near when the products are computed)
    int32_t const j0    = min(base + first * filter64::kGroup + G * (lane & 31), params.count - 1);
    uint32_t const near = *reinterpret_cast<const uint32_t*>(lane < 32 ? params.a + j0 : params.b + j0);
    int32_t const last = (params.count - 1) / filter64::kGroup;
    uint32_t pieces[G][2][6];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      filter64::Group const& from = params.groups[min(base / filter64::kGroup + first + g, last)];
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int d = 0; d < 6; ++d) pieces[g][k][d] = from.pieces[k][d][lane];
    }
    filter64::Sums start;
#pragma unroll
    for (int r = 0; r < 16; ++r) start[r] = filter64::kStart;
    asm("" : "+v"(start));  // (one set of registers, not one filled anew for every block)
    int const scale[2] = {filter64::scale_of(0, lane), filter64::scale_of(1, lane)};
    Ranked ranked[G];
#pragma unroll
    for (int g = 0; g < G; ++g) ranked[g] = Ranked{kNoKey, kNoKey, kNoKey};
    uint32_t half_block = static_cast<uint32_t>(lane) >> 5;
    for (uint32_t i = 0; i < count; i += 32u, half_block += 2u) {
      filter64::V8 const digits = filter64::digits_of(hashes[i + static_cast<uint32_t>(lane % 32)]);
#pragma unroll
      for (int g = 0; g < G; ++g) ranked[g].add(filter64::least_of(filter64::sums_of(digits, pieces[g][0], pieces[g][1], scale[0], scale[1], start)) << 16 | half_block);
    }
    asm volatile("" : : "v"(near));
#pragma unroll
    for (int g = 0; g < G; ++g) ranked[g].merge_halves();
#pragma unroll
    for (int g = 0; g < G; g += 2) {
      bool const two = g + 1 < G;
      settle(ranked[g], ranked[two ? g + 1 : g], (first + g) * filter64::kGroup + (two ? lane : lane % filter64::kGroup), two, hashes, count);
    }
  }

  // hashes: `count` of them, and room up to the next multiple of 32.  They are left to gather until kFoldFrom are there.
  __device__ __forceinline__ uint32_t fold(T* hashes, uint32_t count, bool last)
  {
    if (count < kFoldFrom && !last) return count;
    if (count == 0) return 0;
    wave_lds_fence();
    // (a hash that is there twice does not change a minimum)
    uint32_t const rest = (0u - count) & 31u;
    if (static_cast<uint32_t>(lane) < rest) hashes[count + lane] = hashes[0];
    wave_lds_fence();
    if (kCutUp && AT_ONCE != kLeast && groups == kLeast) {
      fold_groups<kLeast>(0, hashes, count + rest);
    } else {
#pragma unroll 1
      for (int g = 0; g + AT_ONCE <= groups; g += AT_ONCE) fold_groups<AT_ONCE>(g, hashes, count + rest);
      if constexpr (GROUPS % AT_ONCE != 0) {
        if (groups == GROUPS) fold_groups<GROUPS % AT_ONCE>(GROUPS / AT_ONCE * AT_ONCE, hashes, count + rest);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return 0;
  }
  __device__ __forceinline__ void finish() { wave_lds_fence(); }
  template <typename Put>
  __device__ __forceinline__ void each(Put const& put) const
  {
    for (int j = lane; j < slots(); j += kWave) put(j, lds->minima[j]);
    __builtin_amdgcn_wave_barrier();
  }
  static constexpr uint32_t kNoKey = 0xFFFFFFFFu;
};

// Puts the fresh ones of a trip's hashes (a lane with `valid` has one) behind the `count` that wait in lds.hashes: those that
// the wavefront has not met lately.
template <int N>
__device__ __forceinline__ void gather(WaveLds<uint32_t>& lds, bool const (&valid)[N], uint32_t const (&hv)[N], uint32_t* count)
{
#pragma unroll
  for (int n = 0; n < N; ++n) {
    bool fresh = false;
    if (valid[n]) {
      uint32_t* const at = &lds.recent[hv[n] & (kRecentEntries - 1)];
      fresh              = *at != hv[n];
      *at                = hv[n];
    }
    uint64_t const vm = ballot64(fresh);
    if (fresh) lds.hashes[*count + lanes_below(vm)] = hv[n];
    *count += static_cast<uint32_t>(__builtin_popcountll(vm));
  }
}
// 64-bit hashes: the table says where among the hashes that were gathered (and perhaps folded since, in the same part) it may be
template <int N>
__device__ __forceinline__ void gather(WaveLds<uint64_t>& lds, bool const (&valid)[N], uint64_t const (&hv)[N], uint32_t* count)
{
  // (one after the other: the second of a lane's windows finds those of the first, 20,011 long rows 2759 -> 2711 us)
#pragma unroll
  for (int n = 0; n < N; ++n) {
    uint16_t* const at = &lds.recent[static_cast<uint32_t>(hv[n]) & (kRecentEntries - 1)];
    uint64_t const vm  = ballot64(valid[n]) & ballot64(lds.hashes[*at] != hv[n]);  // (no branch: recent holds places of hashes, for whatever hv; 20,011 long rows 2704 -> 2689 us)
    if (__builtin_amdgcn_inverse_ballot_w64(vm)) {
      uint32_t const place = *count + lanes_below(vm);
      lds.hashes[place]    = hv[n];
      *at                  = static_cast<uint16_t>(place);
    }
    *count += static_cast<uint32_t>(__builtin_popcountll(vm));
  }
}
template <typename T>
__device__ __forceinline__ void forget_hashes(WaveLds<T>& lds, int lane)
{
  // (0 is no hash; a place of 64-bit hashes is the one behind all others, which holds 0)
  uint32_t const none = sizeof(T) == 4 ? 0u : kNoPlace * 0x10001u;
  if (sizeof(T) == 8 && lane == 0) lds.hashes[kNoPlace] = 0;
#pragma unroll
  for (int i = 0; i < static_cast<int>(sizeof(lds.recent) / 16); i += kWave) reinterpret_cast<uint4*>(lds.recent)[i + lane] = make_uint4(none, none, none, none);
}

// What is hashed: a column of strings, by windows of characters, or a column of lists of strings, by runs of elements.  A
// row's length is what it is cut by (bytes; positions of runs), and process() folds the hashes of the part [begin, end) of
// row i into the minima.
template <typename T_>
struct TextRows {
  using T   = T_;
  using Lds = WaveLds<T>;
  static constexpr const char* kName = "minhash_parts_kernel";
  static constexpr bool kShortRows   = false;  // no more is known of their lengths than the kernels read
  // groups of 64-bit parameters at a time where there are six and more, whose minima leave LDS for three workgroups only: four
  // (30,000 rows of 3000 bytes, 200 parameters: two 1709 us, three 1780, four 1631)
  static constexpr int kManyGroups   = 4;
  static constexpr int kSimdWaves   = sizeof(T) == 4 ? 6 : 4;  // wavefronts per SIMD that its LDS leaves room for
  // (parts of up to one and a half of it.  The end of the kernel is uneven by one of them; what a part costs beside its
  // length is little with 32-bit hashes, for which 4096 is no faster, and a twentieth with 64-bit ones: 60,000 rows of
  // 14,000 bytes, 128 parameters: 2816: 13.07 ms, 4096: 12.87, 6144: 12.99, which loses 3 % where rows are shorter)
  static constexpr int64_t kPart    = sizeof(T) == 4 ? 2816 : 4096;
  static constexpr int64_t kMinPart = kTile;  // less would be staged for its halo
  static constexpr int kPartCost    = 64;
  ColView col;
  T seed;
  int32_t width;

  __device__ __forceinline__ int32_t rows() const { return col.size; }
  __device__ __forceinline__ bool masked() const { return col.use_mask; }
  __device__ __forceinline__ bool valid(int64_t i) const { return col.valid(i); }
  __device__ __forceinline__ int64_t length(int64_t i) const { return col.off(i + 1) - col.off(i); }
  __device__ __forceinline__ int64_t total() const { return col.off(col.size) - col.off(0); }
  template <typename Minima>
  __device__ __forceinline__ void process(int64_t i, int64_t begin, int64_t end, Minima& minima, Lds& lds, int lane) const
  {
    using H              = HashTraits<T>;
    int64_t const o          = col.off(i);
    int64_t const left       = col.off(i + 1) - o - begin;  // bytes from the part's first to the row's last
    const uint8_t* const row = col.chars + o + begin;
    int32_t const span       = static_cast<int32_t>(end - begin);
    forget_hashes(lds, lane);  // (the wave barrier after the first tile's staging comes before the first look)
    uint32_t count = 0;        // hashes that wait to be folded (wave-uniform)
    // usual case: a window (<= 4*width bytes) fits the halo staged behind every tile
    bool const narrow = static_cast<int64_t>(width) * 4 <= kHalo;
    int32_t const n   = static_cast<int32_t>(min(left, static_cast<int64_t>(1) << 30));
    auto const starts_at = [&](int32_t base) { return static_cast<uint32_t>(min(kTile, span - base)); };
    TileBytes tile;  // asked for a tile ahead
    auto const fetch = [&](int32_t base) { tile.fetch(row + base, tile_length(n, base, starts_at(base), width), lane); };
    if (narrow) fetch(0);
    for (int32_t base = 0; base < span;) {
      if (narrow) {
        uint32_t const cnt = starts_at(base);
        auto const hash    = [seed = seed](auto const& src, uint32_t len, auto& h) { H::hash(src, len, seed, h); };
        auto const next    = [&] {
          if (base + kTile < span) fetch(base + kTile);
        };
        hash_tile_windows<T>(tile, next, row, n, left - n, begin == 0, base, cnt, width, lds.bytes, lds.chars, lane, hash,
                             [&](auto const& valid, auto const& hv) { gather(lds, valid, hv, &count); });
        base += kTile;
      } else {
        // very wide windows: 64 starts at a time, bytes read straight from global memory
        int32_t const pos = base + lane;
        bool valid        = false;
        T hv[1]           = {0};
        if (pos < span) {
          int64_t const remaining = left - pos;
          BoundedSrc const src[1] = {{row + pos, remaining}};
          uint32_t hlen;
          uint32_t const readable = static_cast<uint32_t>(min(remaining, static_cast<int64_t>(width) * 4));
          valid = window_at(src[0], row + pos, remaining, readable, begin == 0 && pos == 0, false, width, &hlen);
          if (valid) H::hash(src, hlen, seed, hv);
        }
        uint64_t const vm = ballot64(valid);
        if (valid) lds.hashes[count + lanes_below(vm)] = hv[0];
        count += static_cast<uint32_t>(__builtin_popcountll(vm));
        base += kWave;
      }
      count = minima.fold(lds.hashes, count, base >= span);
    }
  }
};

struct ListView {
  const int32_t* offsets;  // element index of the first element of row i + offset
  const uint32_t* mask;
  int32_t size;
  int32_t offset;
  int32_t use_mask;
  ColView child;           // the elements

  __device__ __forceinline__ int64_t off(int64_t i) const { return offsets[i + offset]; }
  __device__ __forceinline__ bool valid(int64_t i) const
  {
    if (!use_mask) return true;
    int64_t const b = i + offset;
    return (mask[b >> 5] >> (b & 31)) & 1u;
  }
};

// Byte source over global memory through aligned dword loads that overlap [p, p + len) only.
struct AlignedSrc {
  static constexpr bool kInTile = false;
  const uint32_t* w;  // aligned address at or below the first byte
  uint32_t mis;       // first byte inside w[0]
  uint32_t end;       // mis + len
  __device__ __forceinline__ AlignedSrc(const uint8_t* p, uint32_t len)
  {
    mis = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p) & 3u);
    w   = reinterpret_cast<const uint32_t*>(p - mis);
    end = mis + len;
  }
  __device__ __forceinline__ uint32_t byte(uint32_t i) const { return reinterpret_cast<const uint8_t*>(w)[mis + i]; }
  __device__ __forceinline__ uint32_t dword(uint32_t k) const
  {
    uint32_t const lo = 4u * k < end ? w[k] : 0u;
    uint32_t const hi = 4u * (k + 1u) < end ? w[k + 1] : 0u;
    return __builtin_amdgcn_alignbit(hi, lo, mis * 8u);
  }
};

constexpr uint32_t kRunStageBytes = 4096;                           // longest stretch of chars hashed out of LDS
constexpr uint32_t kRunStageWords = (kRunStageBytes + 16 + 32) / 4;  // + misalignment, + whole blocks and over-read of the hash tail
template <typename T>
constexpr uint32_t run_hashes() { return sizeof(T) == 4 ? 256 : 512; }  // hashes folded together

template <typename T>
struct RunLds {
  alignas(16) T hashes[run_hashes<T>() + kWave];  // (padded to the stride of the fold, at most 63 more)
  // the chars of the elements a wavefront is hashing (32-bit hash only: measured 13 % faster there, 9 % slower for the
  // 64-bit hash, whose 16-byte steps cost more to assemble out of LDS than they save)
  alignas(16) uint32_t bytes[sizeof(T) == 4 ? kRunStageWords : 4];
};

// The runs of elements of minhash_ngrams (cpp/src/text/minhash.cu:182-250).  Positions are list elements, 64 a trip; the hashes of up to four trips are folded together.
template <typename T_>
struct RunRows {
  using T   = T_;
  using Lds = RunLds<T>;
  static constexpr const char* kName = "minhash_ngrams_parts_kernel";
  static constexpr bool kShortRows   = true;
  static constexpr int kManyGroups   = 2;  // (four wavefronts: 20,000 lists of 480, 256 parameters 363 us, with three and four groups 405)
  static constexpr int kSimdWaves   = sizeof(T) == 4 ? 7 : 5;
  static constexpr int64_t kPart    = 704;
  static constexpr int64_t kMinPart = kWave;
  static constexpr int kPartCost    = 32;
  ListView col;
  T seed;
  int32_t ngrams;

  __device__ __forceinline__ int32_t rows() const { return col.size; }
  __device__ __forceinline__ bool masked() const { return col.use_mask; }
  __device__ __forceinline__ bool valid(int64_t i) const { return col.valid(i); }
  // minhash.cu:311-314 with width = ngrams: the positions that the permutation looks at
  __device__ __forceinline__ int64_t length(int64_t i) const
  {
    int64_t const n = col.off(i + 1) - col.off(i);
    return n == 0 ? 0 : max(static_cast<int64_t>(1), n - ngrams + 1);
  }
  __device__ __forceinline__ int64_t total() const { return col.off(col.size) - col.off(0); }
  template <typename Minima>
  __device__ __forceinline__ void process(int64_t i, int64_t begin, int64_t end, Minima& minima, Lds& lds, int lane) const
  {
    using H             = HashTraits<T>;
    int64_t const first = col.off(i);
    int64_t const n     = col.off(i + 1) - first;
    // the bytes from the start of the lane's element to the end of the last element of its run (224-229), clamped to the
    // row (218-222); asked for a trip ahead
    int64_t bo, eo;
    auto const ask = [&](int64_t base) {
      int64_t const idx = min(base + lane, n - 1);
      bo                = col.child.off(first + idx);
      eo                = col.child.off(first + min(idx + ngrams, n - 1) + 1);
    };
    ask(begin);
    uint32_t count = 0;
    for (int64_t base = begin; base < end; base += kWave) {
      int64_t const idx = base + lane;
      // a clamped run counts only at element 0 (218-222); a null element starts no run (213-216)
      bool const valid        = idx < end && (idx == 0 || idx + ngrams < n) && col.child.valid(first + idx);
      int64_t const run_begin = bo;
      uint32_t const run      = static_cast<uint32_t>(eo - bo);
      T hv[1]                 = {0};
      // The runs of these 64 elements overlap and lie side by side in the chars: fetch that stretch once, with
      // coalesced loads, and hash out of LDS (the hash walks a run dword by dword, each step a dependent read).
      // A stretch too long for the buffer is hashed straight from memory.
      int64_t const span_begin = static_cast<int64_t>(wave_bcast64(static_cast<uint64_t>(bo), 0));
      int64_t const span_end   = static_cast<int64_t>(wave_bcast64(static_cast<uint64_t>(eo), kWave - 1));
      if (base + kWave < end) ask(base + kWave);
      if (sizeof(T) == 4 && span_end - span_begin <= static_cast<int64_t>(kRunStageBytes)) {
        uint32_t const mis = stage_bytes(col.child.chars, span_begin, static_cast<uint32_t>(span_end - span_begin), lds.bytes, lane);
        wave_lds_fence();
        WordSrc const src[1] = {WordSrc(lds.bytes, mis + static_cast<uint32_t>(run_begin - span_begin))};
        if (valid) H::hash(src, run, seed, hv);
        wave_lds_fence();
      } else if (valid) {
        AlignedSrc const src[1] = {AlignedSrc(col.child.chars + run_begin, run)};
        H::hash(src, run, seed, hv);
      }
      uint64_t const vm = ballot64(valid);
      if (valid) lds.hashes[count + lanes_below(vm)] = hv[0];
      count += static_cast<uint32_t>(__builtin_popcountll(vm));
      if (count > run_hashes<T>() - kWave) {  // (whole blocks but where elements are null)
        minima.fold(lds.hashes, count, true);
        count = 0;
      }
    }
    minima.fold(lds.hashes, count, true);
  }
};

// How the rows are shared out: every row is cut into parts of about one length, the parts are numbered row after row
// (prefix), and a wavefront takes a unit of work, a few consecutive parts, at a time.
template <typename Source>
struct RowParts {
  Source source;
  int32_t waves;  // wavefronts that the device holds
  int32_t least;  // the least part: Source::kMinPart, more where the products of a row are computed exactly at its end
  // What every wavefront has to do.
  __device__ __forceinline__ int64_t share() const
  {
    return static_cast<int64_t>(static_cast<double>(source.total()) / waves);  // (whole division of 64 bits: a hundred instructions)
  }
  // Length of a part: kPart where that leaves every wavefront four parts and more, else a quarter of what each has to
  // do, in columns of less than four of the smallest parts per wavefront half of it (20,000 rows of 300 bytes, 64
  // parameters: the whole share 60 us, half of it 52, a quarter 54; 8,193 lists of 200 elements, 128 parameters: 42, 39,
  // 45).  Parts of a row of length n that is not null: as many as come nearest to the length, so that none is a remainder
  // (a row of up to one and a half stays whole), but in a column of fewer rows than wavefronts, where some would be left
  // without work, as many as keep each within the length (5,000 lists of 130 elements: 23.6 us, the nearest 25.4).  An
  // empty row has one (its zeros have to be written).  Any number from one to the row's trips will do: what a division
  // would give is not needed.
  struct Cut {
    float per_length, more;
  };
  __device__ __forceinline__ Cut cut() const
  {
    int64_t const all    = share();
    int64_t const length = (all / (all < 4 * Source::kMinPart ? 2 : 4) + kWave) / kWave * kWave;
    float const within   = static_cast<float>(min(max(length, static_cast<int64_t>(least)), Source::kPart));
    return Cut{__builtin_amdgcn_rcpf(within), source.rows() <= waves ? within - 1.0f : within / 2.0f};
  }
  __device__ __forceinline__ uint32_t parts_of(int64_t n, Cut const& c) const
  {
    return max(1u, static_cast<uint32_t>((static_cast<float>(n) + c.more) * c.per_length));
  }
  // Part i of k of a row of length n: whole trips of 64 (of 256, four of which are staged or folded together, where a part
  // has several of those), as even as they come.  A row has at least as many trips as parts.
  __device__ __forceinline__ void bounds(int64_t n, uint32_t i, uint32_t k, int64_t* begin, int64_t* end) const
  {
    *begin = 0;
    *end   = n;
    if (k == 1) return;
    uint32_t const trip  = n >= static_cast<int64_t>(k) * 1024 ? 256u : 64u;
    uint64_t const trips = static_cast<uint64_t>(n + trip - 1) / trip;
    uint64_t const each  = trips >> 32 ? trips / k : static_cast<uint32_t>(trips) / k;
    uint32_t const more  = static_cast<uint32_t>(trips - each * k);
    *begin = static_cast<int64_t>(trip * (each * i + min(i, more)));
    *end   = min(n, *begin + static_cast<int64_t>(trip * (each + (i < more ? 1u : 0u))));
  }
  // Parts to a unit: an eighth of the parts there are for a wavefront, and no more than make up kPart (with what a part
  // costs beside its length); and whether one counter keeps up with handing the units out.  It answers 150 M requests a
  // second, and a position costs about one instruction for its hash and 1.5 for every 64 parameters (64-bit hashes: four
  // and 2.5): one counter where a unit takes some 8192, which is twice what the device gets through meanwhile.  (Of
  // 131,071 rows of 3000 bytes, 260 parameters, 32 groups with a counter each took 4.57 ms, one counter 4.42: the groups
  // are not done at one time.  With 26 parameters one counter took 2.10 ms, 32 took 1.25.)
  __device__ __forceinline__ uint32_t per_unit(uint32_t total, int32_t params, bool* one_counter) const
  {
    float const mean    = static_cast<float>(source.total()) * __builtin_amdgcn_rcpf(static_cast<float>(max(total, 1u)));
    uint32_t const most = static_cast<uint32_t>(static_cast<float>(Source::kPart) * __builtin_amdgcn_rcpf(mean + static_cast<float>(Source::kPartCost)));
    uint32_t const each = max(1u, min(total / (8u * static_cast<uint32_t>(waves)), most));
    float const work    = sizeof(typename Source::T) == 4 ? static_cast<float>(43 + params) / 43.0f : static_cast<float>(100 + params) / 25.0f;
    *one_counter        = mean * static_cast<float>(each) * work >= 8192.0f;
    return each;
  }
};

// Wavefronts per SIMD that the kernels are compiled for.
template <typename Source, typename Minima>
constexpr int simd_waves()
{
  // (as many workgroups to a CU; LDS is given out in pieces of 1280 bytes)
  constexpr int kPiece = 1280, kPieces = (kWaves * static_cast<int>(sizeof(typename Source::Lds) + sizeof(typename Minima::Lds)) + kPiece - 1) / kPiece;
  return std::min({Source::kSimdWaves, Minima::kSimdWaves, 160 * 1024 / kPiece / kPieces});
}

// The row r that part t is one of, prefix[r] <= t < prefix[r + 1], is one of 64 rows from the returned one on, of which
// *near is prefix (rows + 1 of them), a lane a row; not the last.  Looked for first where rows of equal numbers of parts
// would have it, then where the parts missing from there would lie, then with 64 rows to a step.
__device__ __forceinline__ int64_t row_of(const uint32_t* __restrict__ prefix, int64_t rows, uint32_t total, uint32_t t, int lane, uint32_t* near)
{
  float const slope = static_cast<float>(rows) * __builtin_amdgcn_rcpf(static_cast<float>(total));
  int64_t guess     = static_cast<int64_t>(static_cast<float>(t) * slope);
#pragma unroll 1
  for (int probe = 0; probe < 2; ++probe) {
    int64_t const from  = __builtin_amdgcn_readfirstlane(static_cast<int>(min(max(guess - kWave / 2, static_cast<int64_t>(0)), rows)));
    *near               = from + lane <= rows ? prefix[from + lane] : 0xFFFFFFFFu;
    uint64_t const upto = ballot64(*near <= t);
    if (upto != 0 && upto != ~0ull) return from;
    int32_t const ahead = static_cast<int32_t>(t - wave_bcast(*near, kWave / 2));
    guess += static_cast<int64_t>(static_cast<float>(ahead) * slope);
  }
  int64_t r = 0, end = rows;
  while (end - r > 1) {
    int64_t const step = (end - r + kWave - 1) / kWave;
    int64_t const at   = r + lane * step;
    int const below    = __builtin_popcountll(ballot64(at < end && prefix[min(at, end - 1)] <= t));
    r += (below - 1) * step;
    end = min(end, r + step);
  }
  *near = r + lane <= rows ? prefix[r + lane] : 0xFFFFFFFFu;
  return r;
}

// The parts of a row of so many look at its slots before they ask for a minimum there: an address answers one request at a time,
// which is what one long row took most of its time with, and of thousands of parts a dozen lower a slot.  (What is read may be
// larger than what is there by then, never smaller.)  One row of 3 MB, 26 parameters of 32 bits 146 -> 51 us, 128 264 -> 107, of 64 bits
// 171 -> 74; a list of 3 million elements, 64 parameters 452 -> 95.  In rows of fewer parts the read is waited for in vain: 40 rows of 300 KB
// (600 parts), 128 parameters 88 -> 114, a row of 500 KB (1950) 53 either way, of 700 KB 71 -> 54.
constexpr uint32_t kCrowd = 2048;

// Part t is one of the row r with prefix[r] <= t < prefix[r + 1].  A row of one part is stored, the parts of the others
// meet with an atomic minimum (their slots hold the largest value before).  A wavefront's first unit is its own number in
// the grid, the following ones come from counters: an address answers about 150 M requests a second, which a column of
// short rows exceeds, so there are thirty-two of them, and rows much shorter than a wavefront's share are asked for several at
// a time (131,071 rows of 300 bytes, 64 parameters: one counter and a request a row 1621 us).  Where the parts
// of a unit lie is read once for 64 rows, a lane each.  The chunks of parameters come one after the other in the same count.
template <typename Source, typename Minima, typename T = typename Minima::T>
__global__ void __launch_bounds__(kThreads, (simd_waves<Source, Minima>())) minhash_parts_kernel(RowParts<Source> parts, Params<T> params, int32_t chunks,
                                                                                    const int32_t* __restrict__ out_offsets,
                                                                                    const uint32_t* __restrict__ prefix,
                                                                                    unsigned long long* __restrict__ counters, T* __restrict__ out)
{
  __shared__ typename Source::Lds lds[kWaves];
  __shared__ typename Minima::Lds minima_lds[kWaves];
  Source const& source  = parts.source;
  int64_t const rows    = source.rows();
  uint32_t const total  = prefix[rows];
  bool one_counter;
  uint32_t const each   = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(parts.per_unit(total, min(params.count, Minima::kSlots), &one_counter))));
  uint32_t const units  = total / each + (total % each != 0 ? 1u : 0u);
  // 64-bit hashes: chunks of two groups of parameters where the wavefronts suffice for that, or else of four (the windows are hashed for each
  // of them, by wavefronts that had nothing to do): 100 rows of 2000 bytes, 128 parameters 21 -> 18 us, 260 parameters, in fours,
  // 32 -> 27; 700 of 300, 256 parameters 31 -> 27;
  // with twice or four times as many units as wavefronts it is no gain: 50 rows of 16 KB 33.2 us whole, 36.4 in chunks of two groups
  int32_t in_chunk_groups = 0;  // 0: as many as the minima are made for
  if constexpr (Minima::kCutUp) {
    if (units <= static_cast<uint32_t>(parts.waves)) {
      uint32_t const waves = static_cast<uint32_t>(parts.waves), whole = static_cast<uint32_t>(chunks);
      uint32_t const groups = static_cast<uint32_t>(params.count + filter64::kGroup - 1) / filter64::kGroup, twos = (groups + 1) / 2, fours = (groups + 3) / 4;
      if (twos > whole && units * twos <= waves)
        in_chunk_groups = 2, chunks = static_cast<int32_t>(twos);
      else if (fours > whole && units * fours <= waves)
        in_chunk_groups = 4, chunks = static_cast<int32_t>(fours);
    }
  }
  uint64_t const all    = static_cast<uint64_t>(units) * static_cast<uint32_t>(chunks);
  int const lane        = lane_id();
  int const wave        = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
  uint32_t const me     = blockIdx.x * kWaves + static_cast<uint32_t>(wave);
  uint32_t chunk        = 0;
  Minima minima(&minima_lds[wave], lane, in_chunk_groups);
  minima.load(params, 0);
  for (uint64_t unit = me; unit < all;) {
    while (unit >= static_cast<uint64_t>(chunk + 1u) * units) minima.load(params, static_cast<int32_t>(++chunk));  // (the next chunk of parameters)
    int32_t const chunk_base = static_cast<int32_t>(chunk) * minima.stride();
    int32_t const in_chunk   = min(minima.slots(), params.count - chunk_base);
    uint32_t t               = static_cast<uint32_t>(unit - static_cast<uint64_t>(chunk) * units) * each;
    uint32_t const t_end     = total - t < each ? total : t + each;
    int64_t base  = 0;  // near: prefix of the rows from there on, a lane a row
    uint32_t near = 0xFFFFFFFFu;
    for (; t < t_end; ++t) {
      uint64_t upto = ballot64(near <= t);
      if (upto == 0 || upto == ~0ull) {
        base = row_of(prefix, rows, total, t, lane, &near);
        upto = ballot64(near <= t);
      }
      int const at         = __builtin_popcountll(upto) - 1;  // (less than 63: the row after that of t begins behind t)
      int64_t const r      = base + at;
      uint32_t const first = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(near), at));
      uint32_t const k     = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(near), at + 1)) - first;
      int64_t const n      = source.length(r);
      int64_t begin, end;
      parts.bounds(n, t - first, k, &begin, &end);
      minima.reset();
      if (begin < end) source.process(r, begin, end, minima, lds[wave], lane);
      minima.finish();
      T* const dst = out + static_cast<int64_t>(out_offsets[r]) + chunk_base;
      if (k < kCrowd) {
        minima.each([&](int32_t j, T v) {
          if (j >= in_chunk) return;
          if (k == 1)
            dst[j] = n > 0 ? v : T{0};  // an empty row is zeros (minhash.cu:318)
          else if (v != std::numeric_limits<T>::max())
            atomicMin(&dst[j], v);
        });
      } else {
        minima.each([&](int32_t j, T v) {
          if (j < in_chunk && v < __hip_atomic_load(&dst[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&dst[j], v);
        });
      }
    }
    if (all <= static_cast<uint64_t>(parts.waves)) break;
    uint32_t const group    = one_counter ? kCounterGroups : me % kCounterGroups;
    unsigned long long next = 0;
    if (lane == 0) next = atomicAdd(&counters[group * kCounterLine], 1ull);
    next = wave_bcast64(next, 0);
    unit = one_counter ? next : next * kCounterGroups + group;
  }
}

// The parameters of 64-bit hashes, laid out for the matrix cores.
constexpr int groups_of(int32_t P) { return (P + filter64::kGroup - 1) / filter64::kGroup; }

// The counters start past the units that the wavefronts take by their place: counter g serves the wavefronts g,
// g + kCounterGroups, .. and hands out the units g, g + kCounterGroups, ..; the one behind them serves all.
__device__ __forceinline__ void start_counters(unsigned long long* counters, int32_t waves)
{
  int const g = static_cast<int>(threadIdx.x);
  if (g <= kCounterGroups) counters[g * kCounterLine] = static_cast<unsigned long long>(g < kCounterGroups ? (waves + kCounterGroups - 1 - g) / kCounterGroups : waves);
}

// The parts of a row in the low half, a valid row in the high half.
template <typename Source>
__device__ __forceinline__ uint64_t parts_and_rows(RowParts<Source> const& parts, typename RowParts<Source>::Cut const& cut, int64_t n, bool valid)
{
  return valid ? parts.parts_of(n, cut) | (1ull << 32) : 0ull;
}

// Everything that comes before the hashing of a column of few rows, in one launch: the first workgroups take 1024 rows each
// and find their parts (and, where some are null, the rows' places in the result), what lies before their rows every one
// counts by itself (one workgroup for all rows was bound by its arithmetic: 8,000 rows of 300 bytes, 64 parameters, 36.2 us
// the call, with this 32.6; up to 1023 rows have a kernel of their own: one that could take eight times as many takes 0.8
// of 15 us longer); `fillers` more write the places where no row is null and fill the result; the wavefronts of
// the workgroups behind them lay out the parameters of 64-bit hashes.
constexpr int kPlanThreads  = 1024;
constexpr int kPlanTiles    = 8;
constexpr int32_t kPlanRows = kPlanThreads * kPlanTiles;
template <int TILES, typename Source, typename T = typename Source::T>
__global__ void __launch_bounds__(kPlanThreads) minhash_plan_kernel(RowParts<Source> parts, Params<T> params, filter64::Group* groups, unsigned tiles,
                                                                    unsigned fillers, int32_t* __restrict__ out_offsets, uint32_t* __restrict__ prefix,
                                                                    unsigned long long* __restrict__ counters, T* __restrict__ out, int64_t out_size)
{
  int32_t const rows = parts.source.rows();
  int32_t const P    = params.count;
  if constexpr (sizeof(T) == 8) {
    if (blockIdx.x >= tiles + fillers) {
      int32_t const group = static_cast<int32_t>((blockIdx.x - tiles - fillers) * (kPlanThreads / kWave) + threadIdx.x / kWave);
      if (group < groups_of(P)) filter64::prepare_group(params.a, params.b, P, group, &groups[group], lane_id());
      return;
    }
  }
  if (blockIdx.x >= tiles) {
    int64_t const first  = static_cast<int64_t>(blockIdx.x - tiles) * kPlanThreads + threadIdx.x;
    int64_t const stride = static_cast<int64_t>(fillers) * kPlanThreads;
    if (!parts.source.masked())
      for (int64_t i = first; i <= rows; i += stride) out_offsets[i] = static_cast<int32_t>(i * P);
    for (int64_t i = first; i < out_size; i += stride) out[i] = std::numeric_limits<T>::max();
    return;
  }
  __shared__ uint64_t lds[kPlanThreads / kWave + 1];
  // all loads in flight together, those of the rows before what depends on the whole column's length
  int64_t n[TILES];
  bool valid[TILES];
#pragma unroll
  for (unsigned k = 0; k < TILES; ++k) {
    n[k]     = 0;
    valid[k] = false;
    if (k <= blockIdx.x) {
      int32_t const i = static_cast<int32_t>(k * kPlanThreads + threadIdx.x);
      n[k]            = parts.source.length(min(i, rows - 1));
      valid[k]        = i < rows && parts.source.valid(min(i, rows - 1));
    }
  }
  if (blockIdx.x == 0) start_counters(counters, parts.waves);
  auto const cut  = parts.cut();
  uint64_t before = 0, mine = 0;
#pragma unroll
  for (unsigned k = 0; k < TILES; ++k) {
    uint64_t const v = parts_and_rows(parts, cut, n[k], valid[k]);
    before += k < blockIdx.x ? v : 0ull;
    mine = k == blockIdx.x ? v : mine;
  }
  uint64_t carry = 0, total;
  if (blockIdx.x > 0) block_exclusive_scan64<kPlanThreads>(before, lds, &carry);
  uint64_t const run = carry + block_exclusive_scan64<kPlanThreads>(mine, lds, &total);
  int32_t const i    = static_cast<int32_t>(blockIdx.x * kPlanThreads + threadIdx.x);
  if (i <= rows) {  // (rows + 1 of them)
    prefix[i] = static_cast<uint32_t>(run);
    if (parts.source.masked()) out_offsets[i] = static_cast<int32_t>(run >> 32) * P;
  }
}

// The same for a column of more rows, in two launches: the sums of tiles of rows (parts in the low half, valid rows in the
// high half; the workgroups behind them lay out the parameters of 64-bit hashes), then, from the sums of the tiles before,
// the places of every row, and the largest value into the slots of the rows that are done in several parts: a wavefront
// fills those of sixteen rows, one after the other (of 64: 8,193 lists of 400 elements, 256 parameters, 83.3 us the call, with this 77.4; 0.6 us more
// where no row is cut).  A tile is `passes` times 256 rows, so that there are at
// most kSumTiles.
inline int32_t sum_passes(int32_t rows) { return (rows - 1) / (kThreads * kSumTiles) + 1; }

template <typename Source, typename T = typename Source::T>
__global__ void __launch_bounds__(kThreads) minhash_sums_kernel(RowParts<Source> parts, Params<T> params, filter64::Group* groups, int32_t tiles, int32_t passes,
                                                                uint64_t* __restrict__ sums)
{
  if constexpr (sizeof(T) == 8) {
    if (static_cast<int32_t>(blockIdx.x) >= tiles) {
      int32_t const group = (static_cast<int32_t>(blockIdx.x) - tiles) * kWaves + static_cast<int32_t>(threadIdx.x / kWave);
      if (group < groups_of(params.count)) filter64::prepare_group(params.a, params.b, params.count, group, &groups[group], lane_id());
      return;
    }
  }
  __shared__ uint64_t lds[kWaves + 1];
  auto const cut = parts.cut();
  uint64_t sum   = 0;
  for (int32_t pass = 0; pass < passes; ++pass) {
    int64_t const i = (static_cast<int64_t>(blockIdx.x) * passes + pass) * kThreads + threadIdx.x;
    if (i < parts.source.rows()) sum += parts_and_rows(parts, cut, parts.source.length(i), parts.source.valid(i));
  }
  uint64_t total;
  block_exclusive_scan64<kThreads>(sum, lds, &total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

constexpr int kPlaceThreads = 1024;  // four wavefronts take the rows, all sixteen fill
template <typename Source, typename T = typename Source::T>
__global__ void __launch_bounds__(kPlaceThreads) minhash_places_kernel(RowParts<Source> parts, int32_t P, int32_t passes, const uint64_t* __restrict__ sums,
                                                                       int32_t* __restrict__ out_offsets, uint32_t* __restrict__ prefix,
                                                                       unsigned long long* __restrict__ counters, T* __restrict__ out)
{
  constexpr int kFill = kThreads / (kPlaceThreads / kWave);  // rows of the tile whose slots a wavefront fills
  __shared__ uint64_t lds[kPlaceThreads / kWave + 1];
  __shared__ uint64_t several[kWaves];
  __shared__ int32_t places[kThreads];
  if (blockIdx.x == 0) start_counters(counters, parts.waves);
  int32_t const rows = parts.source.rows();
  auto const cut     = parts.cut();
  int const tid = static_cast<int>(threadIdx.x), lane = lane_id(), wave = tid / kWave;
  uint64_t mine = 0, carry;
  if (threadIdx.x < blockIdx.x) mine = sums[threadIdx.x];
  static_assert(kSumTiles == kPlaceThreads, "a sum per thread");
  block_exclusive_scan64<kPlaceThreads>(mine, lds, &carry);
  for (int32_t pass = 0; pass < passes; ++pass) {
    int64_t const i  = (static_cast<int64_t>(blockIdx.x) * passes + pass) * kThreads + tid;
    uint64_t const v = tid < kThreads && i < rows ? parts_and_rows(parts, cut, parts.source.length(i), parts.source.valid(i)) : 0ull;
    uint64_t total;
    uint64_t const before = block_exclusive_scan64<kPlaceThreads>(v, lds, &total) + carry;  // (its barriers: the tile before is filled)
    carry += total;
    int32_t const place = parts.source.masked() ? static_cast<int32_t>(before >> 32) * P : static_cast<int32_t>(i * P);
    if (tid < kThreads) {
      if (i <= rows) {
        prefix[i]      = static_cast<uint32_t>(before);
        out_offsets[i] = place;
      }
      places[tid]       = place;
      uint64_t const is = ballot64(static_cast<uint32_t>(v) > 1u);
      if (lane == 0) several[wave] = is;
    }
    __syncthreads();
    uint32_t const word = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(several[wave * kFill / kWave] >> (wave * kFill % kWave))));
    for (uint32_t todo = word & ((1u << kFill) - 1u); todo != 0; todo &= todo - 1) {
      T* const dst = out + places[wave * kFill + __builtin_ctz(todo)];
      for (int32_t j = lane; j < P; j += kWave) dst[j] = std::numeric_limits<T>::max();
    }
  }
}

// How the parameters of 32-bit hashes are shared out: chunks of K sets of 64 (every chunk hashes the windows again, and a lane without
// a parameter still folds), or, for 65 to 288 parameters of which at most 32 lie beyond the last full set, one chunk of
// K full sets and a tail that costs the fold the share `lanes of a tail set / 64` of a set.  Costs in 64ths of a set.
struct Sharing {
  int k;
  bool tail;
};
inline Sharing sharing_for(int32_t P)
{
  Sharing best{1, false};
  int64_t best_cost = std::numeric_limits<int64_t>::max();
  for (int k = 1; k <= 5; ++k) {  // the larger K (fewer hashing passes) on a tie
    int64_t const cost = static_cast<int64_t>((P + k * kWave - 1) / (k * kWave)) * k * kWave;
    if (cost <= best_cost) { best_cost = cost; best = Sharing{k, false}; }
  }
  int const full = P / kWave, rest = P % kWave;
  if (full >= 1 && full <= 4 && rest >= 1 && rest <= 32) {
    int64_t const cost = static_cast<int64_t>(full) * kWave + packing_for(rest).ppad;
    if (cost < best_cost) best = Sharing{full, true};
  }
  return best;
}

// Calls launch(which, chunks) for the minima that serve P parameters, which::type, and the chunks of parameters they take.
template <typename M>
struct Which {
  using type = M;
};
template <typename T, typename Launch>
void with_all_products(int32_t P, Launch const& launch)
{
  Sharing const sh     = sharing_for(P);
  int32_t const chunks = sh.tail ? 1 : (P + sh.k * kWave - 1) / (sh.k * kWave);
  switch (sh.k * 2 + (sh.tail ? 1 : 0)) {
    case 10: launch(Which<MinimaAll<T, 5, false>>{}, chunks); break;
    case 9: launch(Which<MinimaAll<T, 4, true>>{}, chunks); break;
    case 8: launch(Which<MinimaAll<T, 4, false>>{}, chunks); break;
    case 7: launch(Which<MinimaAll<T, 3, true>>{}, chunks); break;
    case 6: launch(Which<MinimaAll<T, 3, false>>{}, chunks); break;
    case 5: launch(Which<MinimaAll<T, 2, true>>{}, chunks); break;
    case 4: launch(Which<MinimaAll<T, 2, false>>{}, chunks); break;
    case 3: launch(Which<MinimaAll<T, 1, true>>{}, chunks); break;
    default: launch(Which<MinimaAll<T, 1, false>>{}, chunks); break;
  }
}
// Up to nine groups of 32 parameters in one chunk (every chunk hashes the windows again), beyond that chunks of equal size of
// at most eight.
constexpr int32_t chunks_of(int groups) { return groups <= 9 ? 1 : (groups + 7) / 8; }
template <typename Source, typename Launch>
void with_minima(int32_t P, bool short_rows, Launch const& launch)
{
  using T = typename Source::T;
  if constexpr (sizeof(T) == 4) {
    with_all_products<T>(P, launch);
  } else {
    if constexpr (Source::kShortRows) {
      if (short_rows) return with_all_products<T>(P, launch);
    }
    int const groups     = groups_of(P);
    int32_t const chunks = chunks_of(groups);
    switch ((groups + chunks - 1) / chunks) {
      case 1: launch(Which<Minima64<1, 1>>{}, chunks); break;
      case 2: launch(Which<Minima64<2, 2>>{}, chunks); break;
      case 3: launch(Which<Minima64<3, 2>>{}, chunks); break;
      case 4: launch(Which<Minima64<4, 2>>{}, chunks); break;
      case 5: launch(Which<Minima64<5, 2>>{}, chunks); break;
      case 6: launch(Which<Minima64<6, Source::kManyGroups>>{}, chunks); break;
      case 7: launch(Which<Minima64<7, Source::kManyGroups>>{}, chunks); break;
      case 8: launch(Which<Minima64<8, Source::kManyGroups>>{}, chunks); break;
      default: launch(Which<Minima64<9, Source::kManyGroups>>{}, chunks); break;
    }
  }
}

// Rows of 64-bit hashes shorter than this on average have all their products computed whole.  In units of what a hash and 64
// parameters cost whole: hash and 32 parameters on the matrix cores 0.225, a chunk of parameters that hashes the row again
// 0.5 an element, a pair of groups 36 a row for what is computed exactly at its end; and where the lanes share out few
// parameters, the hashes of a row are filled up to a whole stride.  131,072 lists of 60 elements (fewer of longer ones, 3 to 6 M
// elements in all), us whole and on the matrix cores: 26 parameters, 60: 181 and 213, 130: 157 and 168, 250: 147 and 150; 64
// parameters, 60: 213 and 228, 130: 194 and 177; 128 parameters, 30: 227 and 328, 60: 286 and 298, 130: 278 and 218, 250: 272 and
// 183; 256 parameters, 60: 239 and 236, 130: 240 and 165; 260 parameters, 15: 607 and 691, 30: 499 and 471, 60: 339 and 286.
inline double short_row_length(int32_t P)
{
  Sharing const sh     = sharing_for(P);
  int32_t const chunks = sh.tail ? 1 : (P + sh.k * kWave - 1) / (sh.k * kWave);
  Packing const few    = packing_for(sh.tail ? P - sh.k * kWave : P);
  double const sets    = sh.tail || P <= 32 ? (sh.tail ? sh.k : 0) + few.ppad / 64.0 : static_cast<double>(chunks * sh.k);
  int const groups     = groups_of(P);
  double const spared  = sets - 0.225 * groups - 0.5 * (chunks_of(groups) - chunks);
  return spared > 0.0 ? 36.0 * ((groups + 1) / 2) / spared - few.groups * static_cast<double>(kFoldTrip) : std::numeric_limits<double>::max();
}

// The launches of one minhash call: the places of the rows in the result and their parts, then the hashing kernel.
// prefix holds rows + 1 values, plan kPlanBytes; laid_out (64-bit hashes) groups_of(P).
template <typename Source, typename T = typename Source::T>
void run_minhash(Source const& source, int32_t rows, bool short_rows, const T* a, const T* b, int32_t P, int32_t* offsets, T* child, int64_t child_size,
                 uint32_t* prefix, uint64_t* plan, filter64::Group* laid_out, hipStream_t stream)
{
  int waves = 0;
  with_minima<Source>(P, short_rows, [&](auto which, int32_t) { waves = simd_waves<Source, typename decltype(which)::type>(); });
  // Runs of elements on the matrix cores: a part ends with exact products, which 64 runs are too few for (200 lists of 2500 elements,
  // 256 parameters: parts of 64 and more 51 us, of 128 and more 41; 500 of them 65 and 61).
  int32_t const least = static_cast<int32_t>(Source::kMinPart) * (sizeof(T) == 8 && !short_rows && Source::kMinPart == kWave ? 2 : 1);
  RowParts<Source> const parts{source, device_cus() * 4 * waves, least};
  Params<T> const params{a, b, P, laid_out};
  auto* const counters = reinterpret_cast<unsigned long long*>(plan);
  auto const layers    = [&](int threads) { return laid_out ? (groups_of(P) + threads / kWave - 1) / (threads / kWave) : 0; };
  if (rows < kPlanRows) {
    int64_t const most     = std::max<int64_t>(child_size, rows + 1);
    unsigned const fillers = static_cast<unsigned>(std::min<int64_t>((most + 4 * kPlanThreads - 1) / (4 * kPlanThreads), 256));
    unsigned const tiles   = static_cast<unsigned>(rows / kPlanThreads + 1);
    auto const plan_rows   = tiles == 1 ? minhash_plan_kernel<1, Source> : minhash_plan_kernel<kPlanTiles, Source>;
    hipLaunchKernelGGL(plan_rows, dim3(tiles + fillers + static_cast<unsigned>(layers(kPlanThreads))), dim3(kPlanThreads), 0, stream, parts, params, laid_out,
                       tiles, fillers, offsets, prefix, counters, child, child_size);
  } else {
    uint64_t* const sums = plan + (kCounterGroups + 1) * kCounterLine;
    int32_t const passes = sum_passes(rows), tiles = (rows - 1) / (kThreads * passes) + 1;
    hipLaunchKernelGGL(HIP_KERNEL_NAME(minhash_sums_kernel<Source>), dim3(static_cast<unsigned>(tiles + layers(kThreads))), dim3(kThreads), 0, stream, parts,
                       params, laid_out, tiles, passes, sums);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(minhash_places_kernel<Source>), dim3(static_cast<unsigned>(rows / (kThreads * passes) + 1)), dim3(kPlaceThreads), 0, stream,
                       parts, P, passes, sums, offsets, prefix, counters, child);
  }

  if (child_size > 0) {
    with_minima<Source>(P, short_rows, [&](auto which, int32_t chunks) {
      using Minima = typename decltype(which)::type;
      ProfileScope ps(Source::kName, stream);
      hipLaunchKernelGGL(HIP_KERNEL_NAME(minhash_parts_kernel<Source, Minima>), dim3(static_cast<unsigned>(parts.waves / kWaves)), dim3(kThreads), 0, stream,
                         parts, params, chunks, offsets, prefix, counters, child);
    });
  }
}

template <typename T>
nvtext_amd_status minhash_impl(const nvtext_amd_strings_column* input, T seed, const T* a, const T* b, int64_t a_count, int64_t b_count,
                               int32_t width, void* stream_, const nvtext_amd_allocator* mr_, nvtext_amd_list_column* out, int32_t type_id)
{
  EntryScope const entry(sizeof(T) == 4 ? "nvtext_amd_minhash" : "nvtext_amd_minhash64");
  if (!input || !out) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null argument");
  *out = nvtext_amd_list_column{};
  // cpp/src/text/minhash.cu:435-446, same order and messages
  if (width < 2) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "Parameter width should be an integer value of 2 or greater");
  if (a_count <= 0) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "Parameters A and B cannot be empty");
  if (a_count != b_count) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "Parameters A and B should have the same number of elements");
  if (static_cast<uint64_t>(input->size) * static_cast<uint64_t>(a_count) >= static_cast<uint64_t>(std::numeric_limits<int32_t>::max()))
    return fail(NVTEXT_AMD_OVERFLOW, "The number of parameters times the number of input rows exceeds the column size limit");
  if (input->size < 0 || input->null_count < 0 || input->null_count > input->size) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "invalid column sizes");
  if (input->null_count > 0 && !input->null_mask) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null_count > 0 requires a null mask");

  hipStream_t stream = static_cast<hipStream_t>(stream_);
  Mr mr{mr_, stream};
  int32_t const rows = input->size;
  int32_t const P    = static_cast<int32_t>(a_count);
  out->child_type    = type_id;
  out->size          = rows;
  out->null_count    = input->null_count;
  out->offsets_size  = rows + 1;
  out->offsets_bytes = static_cast<size_t>(rows + 1) * sizeof(int32_t);
  out->offsets       = static_cast<int32_t*>(mr.allocate(out->offsets_bytes));
  if (!out->offsets) return fail(NVTEXT_AMD_ALLOC_FAILED, "offsets allocation failed");
  if (rows == 0) {  // minhash.cu:449 then 616: zero rows, offsets = [0], empty child
    launch_fill_u32(reinterpret_cast<uint32_t*>(out->offsets), 0u, 1, stream);
    NVTEXT_HIP_TRY_OR(hipGetLastError(), nvtext_amd_list_column_free(out, stream_, mr_));
    return NVTEXT_AMD_SUCCESS;
  }
  out->child_size  = static_cast<int64_t>(rows - input->null_count) * P;
  out->child_bytes = static_cast<size_t>(out->child_size) * sizeof(T);
  if (out->child_bytes) {
    out->child = mr.allocate(out->child_bytes);
    if (!out->child) {
      nvtext_amd_list_column_free(out, stream_, mr_);
      return fail(NVTEXT_AMD_ALLOC_FAILED, "child allocation failed");
    }
  }
  if (input->null_mask) {  // copy_bitmask(input): cpp/src/bitmask/null_mask.cu:381-391
    out->null_mask_bytes = mask_alloc_bytes(rows);
    out->null_mask       = static_cast<uint32_t*>(mr.allocate(out->null_mask_bytes));
    if (!out->null_mask) {
      nvtext_amd_list_column_free(out, stream_, mr_);
      return fail(NVTEXT_AMD_ALLOC_FAILED, "mask allocation failed");
    }
    launch_copy_bitmask(out->null_mask, input->null_mask, input->offset, rows, stream);
  }

  ColView const v = make_view(*input);
  size_t const temp_bytes[3] = {kPlanBytes, static_cast<size_t>(rows + 1) * sizeof(uint32_t),
                                sizeof(T) == 8 ? static_cast<size_t>(groups_of(P)) * sizeof(filter64::Group) : 0};
  TempParts<3> const temp(mr, temp_bytes);
  if (!temp.ok()) {
    nvtext_amd_list_column_free(out, stream_, mr_);
    return fail(NVTEXT_AMD_ALLOC_FAILED, "temporary allocation failed");
  }
  run_minhash(TextRows<T>{v, seed, width}, rows, false, a, b, P, out->offsets, static_cast<T*>(out->child), out->child_size, temp.part<uint32_t>(1),
                 temp.part<uint64_t>(0), temp.part<filter64::Group>(2), stream);
  NVTEXT_HIP_TRY_OR(hipGetLastError(), nvtext_amd_list_column_free(out, stream_, mr_));
  return NVTEXT_AMD_SUCCESS;
}


// ------------------------------------------------------------------ minhash_ngrams / minhash64_ngrams
template <typename T>
nvtext_amd_status minhash_ngrams_impl(const nvtext_amd_list_strings_column* input, int32_t ngrams, T seed, const T* a, const T* b,
                                      int64_t a_count, int64_t b_count, void* stream_, const nvtext_amd_allocator* mr_,
                                      nvtext_amd_list_column* out, int32_t type_id)
{
  EntryScope const entry(sizeof(T) == 4 ? "nvtext_amd_minhash_ngrams" : "nvtext_amd_minhash64_ngrams");
  if (!input || !out) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null argument");
  *out = nvtext_amd_list_column{};
  // cpp/src/text/minhash.cu:524-536, same order and messages
  if (ngrams < 2) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "Parameter ngrams should be an integer value of 2 or greater");
  if (a_count <= 0) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "Parameters A and B cannot be empty");
  if (a_count != b_count) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "Parameters A and B should have the same number of elements");
  if (static_cast<uint64_t>(input->size) * static_cast<uint64_t>(a_count) >= static_cast<uint64_t>(std::numeric_limits<int32_t>::max()))
    return fail(NVTEXT_AMD_OVERFLOW, "The number of parameters times the number of input rows exceeds the column size limit");
  if (input->size < 0 || input->null_count < 0 || input->null_count > input->size) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "invalid column sizes");
  if (input->null_count > 0 && !input->null_mask) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null_count > 0 requires a null mask");
  if (input->size > 0 && !input->offsets) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "a list column with rows needs offsets");
  if (input->child.null_count > 0 && !input->child.null_mask) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null_count > 0 requires a null mask");

  hipStream_t stream = static_cast<hipStream_t>(stream_);
  Mr mr{mr_, stream};
  int32_t const rows = input->size;
  int32_t const P    = static_cast<int32_t>(a_count);
  out->child_type    = type_id;
  out->size          = rows;
  out->null_count    = input->null_count;
  out->offsets_size  = rows + 1;
  out->offsets_bytes = static_cast<size_t>(rows + 1) * sizeof(int32_t);
  out->offsets       = static_cast<int32_t*>(mr.allocate(out->offsets_bytes));
  if (!out->offsets) return fail(NVTEXT_AMD_ALLOC_FAILED, "offsets allocation failed");
  if (rows == 0) {  // minhash.cu:539 then 616
    launch_fill_u32(reinterpret_cast<uint32_t*>(out->offsets), 0u, 1, stream);
    NVTEXT_HIP_TRY_OR(hipGetLastError(), nvtext_amd_list_column_free(out, stream_, mr_));
    return NVTEXT_AMD_SUCCESS;
  }
  out->child_size  = static_cast<int64_t>(rows - input->null_count) * P;
  out->child_bytes = static_cast<size_t>(out->child_size) * sizeof(T);
  if (out->child_bytes) {
    out->child = mr.allocate(out->child_bytes);
    if (!out->child) {
      nvtext_amd_list_column_free(out, stream_, mr_);
      return fail(NVTEXT_AMD_ALLOC_FAILED, "child allocation failed");
    }
  }
  if (input->null_mask) {
    out->null_mask_bytes = mask_alloc_bytes(rows);
    out->null_mask       = static_cast<uint32_t*>(mr.allocate(out->null_mask_bytes));
    if (!out->null_mask) {
      nvtext_amd_list_column_free(out, stream_, mr_);
      return fail(NVTEXT_AMD_ALLOC_FAILED, "mask allocation failed");
    }
    launch_copy_bitmask(out->null_mask, input->null_mask, input->offset, rows, stream);
  }

  ListView v;
  v.offsets  = input->offsets;
  v.mask     = input->null_mask;
  v.size     = rows;
  v.offset   = input->offset;
  v.use_mask = (input->null_mask != nullptr && input->null_count > 0) ? 1 : 0;
  v.child    = make_view(input->child);
  // (a view's child may hold more elements than the view: then the other way is taken, with the same result)
  // Few elements have all their products computed as well, while there are not many of these: the plan need not lay the parameters
  // out.  The lines are where no length of list is slower on the matrix cores (us whole and there: lists of 2500 elements, 256
  // parameters, 160,000 elements 23.4 and 26.9, 260,000 32.1 and 31.1; lists of 150, 512 parameters, 160,000: 39.6 and 44.6; 1024,
  // 90,000: 43.4 and 46.4, 130,000: 55.8 and 56.0, of 2500 52.8 and 47.2; 2048, 60,000: 54.1 and 55.0, of 2500 54.0 and 43.2).
  constexpr int32_t kFewElements = 200000;
  constexpr int64_t kFewProducts = 125000000;
  bool const few        = input->child.size < kFewElements && static_cast<int64_t>(input->child.size) * P < kFewProducts;
  bool const short_rows = sizeof(T) == 8 && (few || static_cast<double>(input->child.size) < short_row_length(P) * rows);
  size_t const temp_bytes[3] = {kPlanBytes, static_cast<size_t>(rows + 1) * sizeof(uint32_t),
                                sizeof(T) == 8 ? static_cast<size_t>(groups_of(P)) * sizeof(filter64::Group) : 0};
  TempParts<3> const temp(mr, temp_bytes);
  if (!temp.ok()) {
    nvtext_amd_list_column_free(out, stream_, mr_);
    return fail(NVTEXT_AMD_ALLOC_FAILED, "temporary allocation failed");
  }
  run_minhash(RunRows<T>{v, seed, ngrams}, rows, short_rows, a, b, P, out->offsets, static_cast<T*>(out->child), out->child_size,
              temp.part<uint32_t>(1), temp.part<uint64_t>(0), short_rows ? nullptr : temp.part<filter64::Group>(2), stream);
  NVTEXT_HIP_TRY_OR(hipGetLastError(), nvtext_amd_list_column_free(out, stream_, mr_));
  return NVTEXT_AMD_SUCCESS;
}

// ------------------------------------------------------------------ minhash without allocations
constexpr int kMaxDevices = 64;
std::mutex g_scratch_lock;
void* g_scratch_ptr[kMaxDevices] = {};

// The address of this device's copy of the array (the array's name means nothing to host code).
nvtext_amd_status scratch_of_current_device(unsigned char** out)
{
  int device = -1;
  NVTEXT_HIP_TRY(hipGetDevice(&device));
  if (device < 0 || device >= kMaxDevices) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "device index out of range");
  std::lock_guard<std::mutex> hold(g_scratch_lock);
  if (!g_scratch_ptr[device]) {
    void* p = nullptr;
    NVTEXT_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[device] = p;
  }
  *out = static_cast<unsigned char*>(g_scratch_ptr[device]);
  return NVTEXT_AMD_SUCCESS;
}

}  // namespace
}  // namespace nvtext_amd

extern "C" {

nvtext_amd_status nvtext_amd_minhash_preallocated(const nvtext_amd_strings_column* input, uint32_t seed, const uint32_t* a, const uint32_t* b,
                                                  int64_t a_count, int64_t b_count, int32_t width, void* stream_, int32_t* out_offsets,
                                                  uint32_t* out_child, int64_t out_child_capacity, uint32_t* out_null_mask)
{
  using namespace nvtext_amd;
  EntryScope const entry("nvtext_amd_minhash_preallocated");
  if (!input || !out_offsets) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null argument");
  if (width < 2) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "Parameter width should be an integer value of 2 or greater");
  if (a_count <= 0) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "Parameters A and B cannot be empty");
  if (a_count != b_count) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "Parameters A and B should have the same number of elements");
  if (input->size < 0 || input->null_count < 0 || input->null_count > input->size) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "invalid column sizes");
  if (static_cast<uint64_t>(input->size) * static_cast<uint64_t>(a_count) >= static_cast<uint64_t>(std::numeric_limits<int32_t>::max()))
    return fail(NVTEXT_AMD_OVERFLOW, "The number of parameters times the number of input rows exceeds the column size limit");
  if (input->null_count > 0 && !input->null_mask) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "null_count > 0 requires a null mask");
  if (input->size > kPreallocatedMaxRows)
    return fail(NVTEXT_AMD_INVALID_ARGUMENT, "more rows than nvtext_amd_minhash_preallocated takes (NVTEXT_AMD_MINHASH_PREALLOCATED_MAX_ROWS)");
  int32_t const rows       = input->size;
  int32_t const P          = static_cast<int32_t>(a_count);
  int64_t const child_size = static_cast<int64_t>(rows - input->null_count) * P;
  if (child_size > out_child_capacity || (child_size > 0 && !out_child)) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "out_child is too small");
  if (input->null_mask && !out_null_mask) return fail(NVTEXT_AMD_INVALID_ARGUMENT, "the input has a null mask: out_null_mask is needed");

  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (rows == 0) {
    launch_fill_u32(reinterpret_cast<uint32_t*>(out_offsets), 0u, 1, stream);
    NVTEXT_HIP_TRY(hipGetLastError());
    return NVTEXT_AMD_SUCCESS;
  }
  unsigned char* base = nullptr;
  nvtext_amd_status const st = scratch_of_current_device(&base);
  if (st != NVTEXT_AMD_SUCCESS) return st;
  uint32_t* const prefix   = reinterpret_cast<uint32_t*>(base);
  uint64_t* const plan     = reinterpret_cast<uint64_t*>(base + kScratchPrefixBytes);

  if (input->null_mask) launch_copy_bitmask(out_null_mask, input->null_mask, input->offset, rows, stream);
  ColView const v = make_view(*input);
  // every value of the scratch that the kernels read is written earlier in this same call: nothing to clear
  run_minhash(TextRows<uint32_t>{v, seed, width}, rows, false, a, b, P, out_offsets, out_child, child_size, prefix, plan, nullptr, stream);
  NVTEXT_HIP_TRY(hipGetLastError());
  return NVTEXT_AMD_SUCCESS;
}

nvtext_amd_status nvtext_amd_minhash(const nvtext_amd_strings_column* input, uint32_t seed, const uint32_t* a, const uint32_t* b, int64_t a_count,
                                     int64_t b_count, int32_t width, void* stream, const nvtext_amd_allocator* mr, nvtext_amd_list_column* out)
{
  return nvtext_amd::minhash_impl<uint32_t>(input, seed, a, b, a_count, b_count, width, stream, mr, out, NVTEXT_AMD_TYPE_UINT32);
}

nvtext_amd_status nvtext_amd_minhash64(const nvtext_amd_strings_column* input, uint64_t seed, const uint64_t* a, const uint64_t* b, int64_t a_count,
                                       int64_t b_count, int32_t width, void* stream, const nvtext_amd_allocator* mr, nvtext_amd_list_column* out)
{
  return nvtext_amd::minhash_impl<uint64_t>(input, seed, a, b, a_count, b_count, width, stream, mr, out, NVTEXT_AMD_TYPE_UINT64);
}

nvtext_amd_status nvtext_amd_minhash_ngrams(const nvtext_amd_list_strings_column* input, int32_t ngrams, uint32_t seed, const uint32_t* a,
                                            const uint32_t* b, int64_t a_count, int64_t b_count, void* stream, const nvtext_amd_allocator* mr,
                                            nvtext_amd_list_column* out)
{
  return nvtext_amd::minhash_ngrams_impl<uint32_t>(input, ngrams, seed, a, b, a_count, b_count, stream, mr, out, NVTEXT_AMD_TYPE_UINT32);
}

nvtext_amd_status nvtext_amd_minhash64_ngrams(const nvtext_amd_list_strings_column* input, int32_t ngrams, uint64_t seed, const uint64_t* a,
                                              const uint64_t* b, int64_t a_count, int64_t b_count, void* stream, const nvtext_amd_allocator* mr,
                                              nvtext_amd_list_column* out)
{
  return nvtext_amd::minhash_ngrams_impl<uint64_t>(input, ngrams, seed, a, b, a_count, b_count, stream, mr, out, NVTEXT_AMD_TYPE_UINT64);
}

}  // extern "C"
