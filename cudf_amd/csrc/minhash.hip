// minhash / minhash64 for gfx950.
//
// Replaces the reference's three-kernel pipeline (cpp/src/text/minhash.cu:87-157 seed
// hashes into a chars-sized temporary, 281-376 permutation kernel re-reading it,
// 390-424 size partitioning) with one fused pass and no chars-sized temporary:
//
//   * a wavefront owns a section of a row.  Per 256-position tile it stages the bytes
//     in LDS (coalesced aligned dword loads), hashes the windows with lanes <-> window
//     starts, and compacts the hashes into LDS;
//   * it then switches to lanes <-> parameters: every lane keeps K (a, b) pairs and
//     K running minima in registers and streams the tile's hashes through LDS
//     broadcast reads, so the inner loop is v_mad_u64_u32 + v_min only;
//   * a wavefront does a row alone, or a part of it: rows are cut into parts of at most 4 KiB (of
//     fewer bytes in a column too small to give every wavefront of the device one of that size),
//     and the parts of a row meet in the result with an atomic minimum;
//   * in a tile with characters of more than one byte the wavefront lists the characters first,
//     so that a lane takes a character and reads its window's length instead of walking to it;
//     hashes that the wavefront has folded lately are dropped (a minimum does not mind).
//
// Null rows get no output slot (the reference drops them with purge_nonempty_nulls,
// minhash.cu:626-628), empty rows are all zeros (minhash.cu:318).
#include "common.cuh"
#include "murmur.cuh"
#include "windows.cuh"

#include <limits>
#include <mutex>
#include <type_traits>

// Scratch of nvtext_amd_minhash_preallocated, the entry point that allocates nothing: the part counts of the
// rows (rows + 1 values) and behind them the tile sums of the scans and the counter of the parts.  Every device holds its own copy of the array
// for as long as the library is loaded (4.2 MB).
constexpr int32_t kPreallocatedMaxRows = NVTEXT_AMD_MINHASH_PREALLOCATED_MAX_ROWS;
constexpr size_t kScratchPrefixBytes   = (static_cast<size_t>(kPreallocatedMaxRows) + 1 + 63) / 64 * 64 * sizeof(uint32_t);
constexpr size_t kScratchScanBytes     = (static_cast<size_t>(kPreallocatedMaxRows) / nvtext_amd::kScanTile + 3) * sizeof(uint64_t);
static __device__ __align__(256) unsigned char scratch[kScratchPrefixBytes + kScratchScanBytes];

namespace nvtext_amd {
namespace {

template <typename T>
struct HashTraits;
template <>
struct HashTraits<uint32_t> {
  template <typename Src>
  static __device__ __forceinline__ uint32_t hash(Src const& src, uint32_t len, uint32_t seed)
  {
    return murmur3_x86_32(src, len, seed);
  }
  // Permutation (minhash.cu:350-351) in uint32 arithmetic: the product and sum wrap mod 2^32, after
  // which "% (2^61-1)" and "& max" change nothing: (hv * a + b), see Fold<uint32_t>.
};
template <>
struct HashTraits<uint64_t> {
  template <typename Src>
  static __device__ __forceinline__ uint64_t hash(Src const& src, uint32_t len, uint64_t seed)
  {
    return murmur3_x64_128_lo(src, len, seed);  // minhash.cu:138: first word of the 128-bit hash
  }
  // Permutation (minhash.cu:350-351): ((hv*a + b) mod 2^64) % (2^61-1), see Fold<uint64_t>.
};

// ((h * a + b) mod 2^64) folded once mod 2^61 - 1, that is (x & p) + (x >> 61) for the 64-bit x: at most p + 7; for two
// hashes and one (a, b).  x = h.lo * a.lo + b is one 64-bit multiply-add; the two cross products, of which only the low
// dwords count, are two more, chained (h.lo * a.hi, then h.hi * a.lo added to it), and their sum goes to the high dword
// of x with a plain 32-bit add, which issues in half the cycles of a multiply or of a three-operand add (left to itself
// the compiler makes them two multiplies and a three-operand add).  The fold is a shift and a mask of that dword and
// one more multiply-add (q * 1 + x) for the carry.  Eight instructions per hash, none that only moves a value.  The
// chained pairs of the two hashes stand interleaved in one block of assembly, so that neither waits for its own first
// half; everything else is left to the compiler, which puts an idle cycle between instructions it cannot see into.
__device__ __forceinline__ void permute_fold_u64_pair(uint64_t h0, uint64_t h1, uint64_t a, uint64_t b, uint32_t one, uint64_t* y0,
                                                      uint64_t* y1)
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

// min of two values below 2^62 in one instruction: such bit patterns are non-negative finite doubles
// (or denormals, which this code object keeps: float_denorm_mode_16_64 = 3), and those order like the
// integers.  An operand that is all ones (the "no hash yet" start value, a NaN pattern) loses to the other.
__device__ __forceinline__ uint64_t min_below_2_62(uint64_t m, uint64_t y)
{
  uint64_t r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(m), "v"(y));
  return r;
}

// Folds the compacted hashes first, first + 1, .. of every `stride` (the count padded to a multiple of the stride)
// into m[K]; lanes <-> parameters.  A wavefront whose lanes all hold different parameters folds every hash
// (first 0, stride = the hashes of one trip); with few parameters the lanes form groups that hold the same
// parameters and fold every other trip each (see Packing).
template <typename T, int K>
struct Fold;

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

template <int K>
struct Fold<uint32_t, K> {
  static constexpr uint32_t kPerTrip = 4;
  static __device__ __forceinline__ void run(const uint32_t* hashes, uint32_t padded, uint32_t first, uint32_t stride,
                                             const uint32_t (&a)[K], const uint32_t (&b)[K], uint32_t (&m)[K])
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
};

template <int K>
struct Fold<uint64_t, K> {
  static constexpr uint64_t p = (1ull << 61) - 1;
  // x mod p for x < 2^64: x = q*2^61 + r with q <= 7, so y = r + q <= p + 7.
  static __device__ __forceinline__ uint64_t fold_once(uint64_t x) { return (x & p) + (x >> 61); }

  // hashes per trip: four (with two, and two and more sets of parameters, the loop issued 3 to 5 % less: fewer
  // independent products between a trip's LDS read and its dependent minima)
  static constexpr uint32_t kPerTrip = 4;
  static __device__ __forceinline__ void run(const uint64_t* hashes, uint32_t padded, uint32_t first, uint32_t stride,
                                             const uint64_t (&a)[K], const uint64_t (&b)[K], uint64_t (&m)[K])
  {
    // Fast pass: the final "subtract p if y >= p" is left out.  y >= p needs the top dword of y to be
    // at least 0x1FFFFFFF (one chance in 2^29 per product), which is tracked with a running maximum;
    // if it ever happens the tile is folded again exactly.  Unreduced values are >= p, above every
    // reduced value, so they can never displace a correct minimum.
    uint32_t top = 0;
    uint32_t one;  // the number 1 where the compiler does not see it: q * one + x stays one multiply-add
    asm("s_mov_b32 %0, 1" : "=s"(one));
    for (uint32_t i = first; i < padded; i += stride) {
      uint64_t h[kPerTrip];
#pragma unroll
      for (uint32_t j = 0; j < kPerTrip; ++j) h[j] = hashes[i + j];
#pragma unroll
      for (int k = 0; k < K; ++k) {
#pragma unroll
        for (uint32_t j = 0; j < kPerTrip; j += 2) {
          uint64_t y0, y1;
          permute_fold_u64_pair(h[j], h[j + 1], a[k], b[k], one, &y0, &y1);
          top               = max(max(top, static_cast<uint32_t>(y0 >> 32)), static_cast<uint32_t>(y1 >> 32));
          m[k]              = min_below_2_62(min_below_2_62(m[k], y0), y1);
        }
      }
    }
    if (ballot64(top >= 0x1FFFFFFFu) != 0) {
      // every lane folds every hash here: a minimum does not mind the hashes of the other sets
      for (uint32_t i = 0; i < padded; ++i) {
        uint64_t const h = hashes[i];
#pragma unroll
        for (int k = 0; k < K; ++k) {
          uint64_t const y = fold_once(h * a[k] + b[k]);
          m[k]             = min(m[k], y >= p ? y - p : y);
        }
      }
    }
  }
};

// The parameters beyond the last full set of 64, when there are at most 32 of them: one more (a, b) pair per lane,
// shared out over sets of lanes as Packing describes, so that they cost the fold a share of a full set (4 parameters
// beyond 256: a sixteenth) instead of a whole one.
template <typename T>
struct TailParams {
  T a[1], b[1], m[1];
  Packing pk;
};
struct NoTail {};

template <typename T, int K, typename Tail = NoTail>
__device__ __forceinline__ void fold_hashes(T* hashes, uint32_t count, const T (&a)[K], const T (&b)[K], T (&m)[K], int lane, Packing pk, Tail& tail)
{
  constexpr bool kHasTail = !std::is_same<Tail, NoTail>::value;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (count == 0) return;
  // a duplicate never changes a minimum
  uint32_t stride = K > 1 ? Fold<T, K>::kPerTrip : pk.stride(Fold<T, K>::kPerTrip);  // a power of two, at most 64
  if constexpr (kHasTail) stride = max(stride, tail.pk.stride(Fold<T, 1>::kPerTrip));
  uint32_t const padded = (count + stride - 1u) & ~(stride - 1u);
  if (lane < static_cast<int>(padded - count)) hashes[count + lane] = hashes[0];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // the usual case keeps the loop counter out of the vector registers
  if (K > 1 || pk.groups == 1)
    Fold<T, K>::run(hashes, padded, 0u, Fold<T, K>::kPerTrip, a, b, m);
  else
    Fold<T, K>::run(hashes, padded, pk.first(lane, Fold<T, K>::kPerTrip), pk.stride(Fold<T, K>::kPerTrip), a, b, m);
  if constexpr (kHasTail)
    Fold<T, 1>::run(hashes, padded, tail.pk.first(lane, Fold<T, 1>::kPerTrip), tail.pk.stride(Fold<T, 1>::kPerTrip), tail.a, tail.b, tail.m);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
template <typename T, int K>
__device__ __forceinline__ void fold_hashes(T* hashes, uint32_t count, const T (&a)[K], const T (&b)[K], T (&m)[K], int lane,
                                            Packing pk = Packing{kWave, 1})
{
  NoTail none;
  fold_hashes<T, K, NoTail>(hashes, count, a, b, m, lane, pk, none);
}

// Whether the wavefront has met this hash lately (it is noted either way).  Called by the lanes that have a hash.
template <typename T>
__device__ __forceinline__ bool seen_lately(WaveLds<T>& lds, T hv)
{
  T* const at  = &lds.recent[static_cast<uint32_t>(hv) & (recent_entries<T>() - 1)];
  T const was  = *at;
  *at          = hv;
  return was == hv;
}
template <typename T>
__device__ __forceinline__ void forget_hashes(WaveLds<T>& lds, int lane)
{
  for (int i = lane; i < recent_entries<T>(); i += kWave) lds.recent[i] = T{0};
}

// Processes the window starts [s_begin, s_end) of one row with one wavefront and folds the
// permuted hashes into m[K].  Lane l owns parameters chunk_base + l + 64*k.
template <typename T, int K, typename Tail>
__device__ __forceinline__ void process_section(const uint8_t* row, int64_t n, int64_t s_begin, int64_t s_end, T seed, int32_t width,
                                                const T (&a)[K], const T (&b)[K], T (&m)[K], WaveLds<T>& lds, int lane, Packing pk, Tail& tail)
{
  using H = HashTraits<T>;
  if (static_cast<int64_t>(width) * 4 <= kHalo) {
    // usual case: a window (<= 4*width bytes) fits the halo staged behind every tile
    forget_hashes(lds, lane);  // (the wave barrier after the first tile's staging comes before the first look)
    for (int64_t base = s_begin; base < s_end; base += kTile) {
      uint32_t const cnt = static_cast<uint32_t>(min(static_cast<int64_t>(kTile), s_end - base));
      uint32_t count     = 0;  // compacted hashes so far (wave-uniform)
      auto const hash    = [seed](WordSrc const& src, uint32_t len) {
        T const hv = H::hash(src, len, seed);
        return hv < 1 ? T{1} : hv;  // minhash.cu:141
      };
      hash_tile_windows<T>(row, n, base, cnt, width, lds.bytes, lds.chars, lane, hash, [&](auto const& valid, auto const& hv) {
        for (auto const& h : hv) {
          bool const fresh  = valid[&h - hv] && !seen_lately(lds, h);
          uint64_t const vm = ballot64(fresh);
          if (fresh) lds.hashes[count + lanes_below(vm)] = h;
          count += static_cast<uint32_t>(__builtin_popcountll(vm));
        }
      });
      fold_hashes<T, K, Tail>(lds.hashes, count, a, b, m, lane, pk, tail);
    }
  } else {
    // very wide windows: 64 starts at a time, bytes read straight from global memory
    for (int64_t base = s_begin; base < s_end; base += kWave) {
      int64_t const gpos = base + lane;
      bool valid         = false;
      T hv               = 0;
      if (gpos < s_end) {
        int64_t const remaining = n - gpos;
        BoundedSrc const src{row + gpos, remaining};
        uint32_t hlen;
        uint32_t const readable = static_cast<uint32_t>(min(remaining, static_cast<int64_t>(width) * 4));
        valid = window_at(src, row + gpos, remaining, readable, gpos == 0, false, width, &hlen);
        if (valid) {
          hv = H::hash(src, hlen, seed);
          hv = hv < 1 ? T{1} : hv;
        }
      }
      uint64_t const vm = ballot64(valid);
      if (valid) lds.hashes[lanes_below(vm)] = hv;
      fold_hashes<T, K, Tail>(lds.hashes, static_cast<uint32_t>(__builtin_popcountll(vm)), a, b, m, lane, pk, tail);
    }
  }
}

template <typename T, int K>
__device__ __forceinline__ void load_params(const T* pa, const T* pb, int32_t P, int32_t chunk_base, int lane, T (&a)[K], T (&b)[K], T (&m)[K])
{
#pragma unroll
  for (int k = 0; k < K; ++k) {
    int32_t const j = chunk_base + lane + kWave * k;
    a[k]            = j < P ? pa[j] : T{0};
    b[k]            = j < P ? pb[j] : T{0};
    m[k]            = std::numeric_limits<T>::max();
  }
}

// How the rows are shared out.  In a column of at least kManyRows rows a wavefront does the rows of up to kPartBytes
// bytes alone, several in turn (minhash_rows_kernel), and the longer ones are cut into parts; in a column of fewer rows
// every row is cut into parts (minhash_parts_kernel), so that the device is full whatever the rows' lengths: 999
// documents of 2 KB (256 parameters) with a workgroup each, and another launch for what lay beyond their first 16 KB,
// took 282 us for 23 us of arithmetic, most of it spent on the longest document; 42 us in parts.  20,011 rows of 16 KB
// (uint64, 128 parameters) 9.0 -> 7.4 ms, the long rows of 400,000 documents of 2 KB 9.7 -> 9.2 ms.
// A workgroup lasts as long as its slowest wavefront, and rows differ in length: with one row per wavefront the others
// waited for the longest of four (8 M rows of about 500 bytes: 88 ms; four rows per wavefront 80 ms, sixteen 77 ms).
// More rows per workgroup mean fewer workgroups, and the column needs them all to fill the device and to even out its
// end: the host asks for as many rows per wavefront (a power of two, at most kMaxRowsPerWave) as leave at least
// kMinRowGroups groups.
constexpr int32_t kManyRows     = 131072;
constexpr int64_t kPartBytes    = 4096;
constexpr int64_t kMinPartBytes = 256;     // a tile: less would be staged for its halo
constexpr int kMaxRowsPerWave   = 16;
constexpr int32_t kMinRowGroups = 16384;  // sixteen times the workgroups that 256 CUs hold at four apiece
inline int rows_per_wave(int32_t rows)
{
  int rpw = 1;
  while (rpw < kMaxRowsPerWave && rows / (2 * rpw * kWaves) >= kMinRowGroups) rpw *= 2;
  return rpw;
}

// The parts of every row: none for a null row and for the rows that minhash_rows_kernel does, one for an empty row (its
// zeros have to be written).
struct RowParts {
  ColView col;
  int32_t waves;      // wavefronts that the device holds
  int64_t row_bytes;  // rows of at most this many bytes are done by minhash_rows_kernel; -1: none is
  // Bytes of a part: kPartBytes where that leaves every wavefront four parts and more, else a quarter of what each has to
  // do, in columns of less than a kilobyte per wavefront all of it (a second round of parts would be longer than the
  // imbalance it removes).
  __device__ __forceinline__ int64_t part_bytes() const
  {
    if (row_bytes >= 0) return kPartBytes;
    int64_t const share = (col.off(col.size) - col.off(0)) / waves;
    int64_t const bytes = ((share < 1024 ? share : share / 4) + kWave) / kWave * kWave;
    return min(max(bytes, kMinPartBytes), kPartBytes);
  }
  __device__ __forceinline__ uint64_t operator()(int64_t i) const
  {
    if (!col.valid(i)) return 0;
    int64_t const n = col.off(i + 1) - col.off(i);
    if (n <= row_bytes) return 0;
    int64_t const bytes = part_bytes();
    return n == 0 ? 1 : static_cast<uint64_t>((n + bytes - 1) / bytes);
  }
};

// The tail of a launch with TAIL: the P - 64 K parameters (1..32) beyond the K full sets of the one chunk.
template <typename T, int K, bool TAIL>
struct TailOf {
  using type = NoTail;
  static __device__ __forceinline__ void load(type&, const T*, const T*, int32_t, int) {}
  static __device__ __forceinline__ void reset(type&) {}
  static __device__ __forceinline__ void finish(type&) {}
  static __device__ __forceinline__ T value(type const&) { return T{0}; }
};
template <typename T, int K>
struct TailOf<T, K, true> {
  using type = TailParams<T>;
  static __device__ __forceinline__ void load(type& t, const T* pa, const T* pb, int32_t P, int lane)
  {
    t.pk            = packing_for(P - K * kWave);
    int32_t const j = K * kWave + t.pk.param_lane(lane);
    t.a[0]          = j < P ? pa[j] : T{0};
    t.b[0]          = j < P ? pb[j] : T{0};
    t.m[0]          = std::numeric_limits<T>::max();
  }
  static __device__ __forceinline__ void reset(type& t) { t.m[0] = std::numeric_limits<T>::max(); }
  static __device__ __forceinline__ void finish(type& t) { t.m[0] = t.pk.combine(t.m[0]); }  // every set of lanes then holds the minima
  static __device__ __forceinline__ T value(type const& t) { return t.m[0]; }
};

// Wavefronts per SIMD that the registers are held to.
template <typename T>
constexpr int minhash_waves() { return sizeof(T) == 4 ? 7 : 4; }

// One workgroup per (group of consecutive rows, parameter chunk): its wavefronts take the group's rows of up to kPartBytes
// bytes one at a time from a counter in LDS, so that the four are done together whatever the rows' lengths; the minima
// go from the registers to the result.  The groups lie along x and, beyond kMaxRowBlocks of them, along z.
template <typename T, int K, bool TAIL>
__global__ void __launch_bounds__(kThreads, minhash_waves<T>()) minhash_rows_kernel(ColView col, T seed, const T* __restrict__ pa, const T* __restrict__ pb,
                                                                int32_t P, int32_t width, const int32_t* __restrict__ out_offsets, T* __restrict__ out,
                                                                int per_wave)
{
  using TailT = TailOf<T, K, TAIL>;
  constexpr int kSets = K + (TAIL ? 1 : 0);
  __shared__ WaveLds<T> lds[kWaves];
  __shared__ uint32_t next_row;

  int const group_rows = per_wave * kWaves;
  int64_t const r0     = (static_cast<int64_t>(blockIdx.z) * gridDim.x + blockIdx.x) * group_rows;
  if (r0 >= col.size) return;
  int const lane           = lane_id();
  int const wave           = threadIdx.x / kWave;
  int32_t const chunk_base = blockIdx.y * (K * kWave);  // (with TAIL there is one chunk)
  int32_t const in_chunk   = min(kSets * kWave, P - chunk_base);
  Packing const pk         = K == 1 ? packing_for(P) : Packing{kWave, 1};
  T a[K], b[K], m[K];
  load_params<T, K>(pa, pb, P, chunk_base, pk.param_lane(lane), a, b, m);
  typename TailT::type tail;
  TailT::load(tail, pa, pb, P, lane);

  int const rows_here = static_cast<int>(min(static_cast<int64_t>(group_rows), col.size - r0));
  if (threadIdx.x == 0) next_row = 0;
  __syncthreads();
  for (;;) {
    int t = 0;
    if (lane == 0) t = static_cast<int>(atomicAdd(&next_row, 1u));
    int const i = __builtin_amdgcn_readfirstlane(t);  // (the same in every lane: what depends on it stays scalar)
    if (i >= rows_here) break;
    if (!col.valid(r0 + i)) continue;
    int64_t const o = col.off(r0 + i);
    int64_t const n = col.off(r0 + i + 1) - o;
    if (n > kPartBytes) continue;
#pragma unroll
    for (int k = 0; k < K; ++k) m[k] = std::numeric_limits<T>::max();
    TailT::reset(tail);
    if (n > 0) process_section<T, K>(col.chars + o, n, 0, n, seed, width, a, b, m, lds[wave], lane, pk, tail);
    if (K == 1) m[0] = pk.combine(m[0]);
    TailT::finish(tail);
    T* const dst = out + static_cast<int64_t>(out_offsets[r0 + i]) + chunk_base;
    // an empty row is zeros (minhash.cu:318)
#pragma unroll
    for (int k = 0; k < K; ++k) {
      int32_t const j = lane + kWave * k;  // (with fewer than 64 parameters the first lanes hold one each, in order)
      if (j < in_chunk) dst[j] = n > 0 ? m[k] : T{0};
    }
    if (TAIL && K * kWave + lane < in_chunk) dst[K * kWave + lane] = n > 0 ? TailT::value(tail) : T{0};
  }
}

// Parts of rows, a wavefront each: part t is one of the row r with prefix[r] <= t < prefix[r + 1].  A row of one part is
// stored, the parts of the others meet with an atomic minimum (their slots hold the largest value before).  With more
// than eight parts for every wavefront they are handed out by a counter, else by place (a counter answers about 150 M
// requests a second: seven thousand wavefronts asking at once would wait 50 us).  The chunks of parameters come one
// after the other in the same count.
template <typename T, int K, bool TAIL>
__global__ void __launch_bounds__(kThreads, minhash_waves<T>()) minhash_parts_kernel(RowParts parts, T seed, const T* __restrict__ pa, const T* __restrict__ pb,
                                                                int32_t P, int32_t width, int32_t chunks, const int32_t* __restrict__ out_offsets,
                                                                const uint32_t* __restrict__ prefix, unsigned long long* __restrict__ counter,
                                                                T* __restrict__ out)
{
  using TailT = TailOf<T, K, TAIL>;
  constexpr int kSets = K + (TAIL ? 1 : 0);
  __shared__ WaveLds<T> lds[kWaves];
  ColView const& col    = parts.col;
  uint32_t const total  = prefix[col.size];
  uint64_t const tasks  = static_cast<uint64_t>(total) * static_cast<uint32_t>(chunks);
  int64_t const bytes   = parts.part_bytes();
  int const lane        = lane_id();
  int const wave        = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
  uint64_t const nwaves = static_cast<uint64_t>(gridDim.x) * kWaves;
  Packing const pk      = K == 1 ? packing_for(P) : Packing{kWave, 1};
  T a[K], b[K], m[K];
  typename TailT::type tail;
  uint32_t chunk = 0;
  load_params<T, K>(pa, pb, P, 0, pk.param_lane(lane), a, b, m);
  TailT::load(tail, pa, pb, P, lane);
  for (uint64_t task = static_cast<uint64_t>(blockIdx.x) * kWaves + wave; task < tasks;) {
    uint32_t const t = static_cast<uint32_t>(task - static_cast<uint64_t>(chunk) * total);
    if (t >= total) {  // the next chunk of parameters
      ++chunk;
      load_params<T, K>(pa, pb, P, static_cast<int32_t>(chunk) * (K * kWave), pk.param_lane(lane), a, b, m);
      continue;
    }
    int32_t const chunk_base = static_cast<int32_t>(chunk) * (K * kWave);
    int32_t const in_chunk   = min(kSets * kWave, P - chunk_base);
    // the last row r with prefix[r] <= t, 64 of them looked at in one step
    int64_t r = 0, end = col.size;
    while (end - r > 1) {
      int64_t const step = (end - r + kWave - 1) / kWave;
      int64_t const at   = r + lane * step;
      int const below    = __builtin_popcountll(ballot64(at < end && prefix[min(at, end - 1)] <= t));
      r += (below - 1) * step;
      end = min(end, r + step);
    }
    int64_t const o   = col.off(r);
    int64_t const n   = col.off(r + 1) - o;
    int64_t const sb  = static_cast<int64_t>(t - prefix[r]) * bytes;
    int64_t const se  = min(n, sb + bytes);
    bool const shared = n > bytes;
#pragma unroll
    for (int k = 0; k < K; ++k) m[k] = std::numeric_limits<T>::max();
    TailT::reset(tail);
    if (sb < se) process_section<T, K>(col.chars + o, n, sb, se, seed, width, a, b, m, lds[wave], lane, pk, tail);
    if (K == 1) m[0] = pk.combine(m[0]);
    TailT::finish(tail);
    T* const dst = out + static_cast<int64_t>(out_offsets[r]) + chunk_base;
    auto const put = [&](int32_t j, T v) {
      if (j >= in_chunk) return;
      if (!shared)
        dst[j] = n > 0 ? v : T{0};  // an empty row is zeros (minhash.cu:318)
      else if (v != std::numeric_limits<T>::max())
        atomicMin(&dst[j], v);
    };
#pragma unroll
    for (int k = 0; k < K; ++k) put(lane + kWave * k, m[k]);
    if (TAIL) put(K * kWave + lane, TailT::value(tail));
    if (tasks <= 8 * nwaves) {
      task += nwaves;
    } else {
      unsigned long long next = 0;
      if (lane == 0) next = atomicAdd(counter, 1ull);
      task = nwaves + wave_bcast64(next, 0);
    }
  }
}

struct ValidTimesP {
  ColView col;
  int32_t P;
  __device__ uint64_t operator()(int64_t i) const { return col.valid(i) ? static_cast<uint64_t>(P) : 0; }
};

__global__ void uniform_offsets_kernel(int32_t* out, int32_t rows, int32_t P)
{
  int64_t const i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i <= rows) out[i] = static_cast<int32_t>(i * P);
}

constexpr int32_t kMaxRowBlocks = 1 << 15;  // groups along x (a launch of 4 M rows, 64 to a group, has two layers along z: the tests reach them)

// The largest value into the slots of the rows that are done in several parts, and 0 into the counter of the parts: a
// wavefront looks at 64 rows and fills those of them one after the other.
template <typename T>
__global__ void __launch_bounds__(kThreads) minhash_clear_kernel(RowParts parts, int32_t P, const int32_t* __restrict__ out_offsets,
                                                                 unsigned long long* __restrict__ counter, T* __restrict__ out)
{
  if (blockIdx.x == 0 && threadIdx.x == 0) *counter = 0;
  int const lane  = lane_id();
  int64_t const r = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  bool const many = r < parts.col.size && parts(r) > 1;
  int64_t const o = many ? out_offsets[r] : 0;
  for (uint64_t todo = ballot64(many); todo != 0; todo &= todo - 1) {
    T* const dst = out + static_cast<int64_t>(wave_bcast64(static_cast<uint64_t>(o), __builtin_ctzll(todo)));
    for (int32_t j = lane; j < P; j += kWave) dst[j] = std::numeric_limits<T>::max();
  }
}

// Everything that comes before the hashing of a column of few rows, in one launch: workgroup 0 counts the parts of the
// rows (and finds the rows' places in the result where some are null), the others write the places where none is and
// fill the result.
constexpr int32_t kPlanRows = kScanSmallTiles * kScanTile;
template <typename T>
__global__ void __launch_bounds__(kScanThreads) minhash_plan_kernel(RowParts parts, int32_t P, int32_t* __restrict__ out_offsets,
                                                                    uint32_t* __restrict__ prefix, unsigned long long* __restrict__ counter,
                                                                    T* __restrict__ out, int64_t out_size)
{
  int32_t const rows = parts.col.size;
  if (blockIdx.x > 0) {
    int64_t const first  = static_cast<int64_t>(blockIdx.x - 1) * kScanThreads + threadIdx.x;
    int64_t const stride = static_cast<int64_t>(gridDim.x - 1) * kScanThreads;
    if (!parts.col.use_mask)
      for (int64_t i = first; i <= rows; i += stride) out_offsets[i] = static_cast<int32_t>(i * P);
    for (int64_t i = first; i < out_size; i += stride) out[i] = std::numeric_limits<T>::max();
    return;
  }
  __shared__ uint64_t lds[kScanThreads / kWave + 1];
  uint64_t carry = 0;  // parts in the low half, valid rows in the high half
  for (int32_t tile = 0; tile < rows; tile += kScanTile) {
    int32_t const base = tile + static_cast<int32_t>(threadIdx.x) * kScanItems;
    uint64_t vals[kScanItems], sum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      bool const in = base + k < rows;
      vals[k]       = in ? parts(base + k) | (static_cast<uint64_t>(parts.col.valid(base + k)) << 32) : 0;
      sum += vals[k];
    }
    uint64_t total;
    uint64_t run = block_exclusive_scan64<kScanThreads>(sum, lds, &total) + carry;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      if (base + k < rows) {
        prefix[base + k] = static_cast<uint32_t>(run);
        if (parts.col.use_mask) out_offsets[base + k] = static_cast<int32_t>(run >> 32) * P;
      }
      run += vals[k];
    }
    carry += total;
  }
  if (threadIdx.x == 0) {
    *counter     = 0;
    prefix[rows] = static_cast<uint32_t>(carry);
    if (parts.col.use_mask) out_offsets[rows] = static_cast<int32_t>(carry >> 32) * P;
  }
}

template <typename T, int K, bool TAIL>
void launch_kernels(RowParts const& parts, T seed, const T* a, const T* b, int32_t P, int32_t width, const int32_t* offsets,
                    const uint32_t* prefix, unsigned long long* counter, T* child, hipStream_t stream)
{
  ColView const& v     = parts.col;
  int32_t const chunks = TAIL ? 1 : (P + K * kWave - 1) / (K * kWave);
  if (v.size >= kManyRows) {
    int const per_wave   = rows_per_wave(v.size);
    int32_t const groups = (v.size + per_wave * kWaves - 1) / (per_wave * kWaves);
    dim3 grid(static_cast<unsigned>(std::min(groups, kMaxRowBlocks)), static_cast<unsigned>(chunks),
              static_cast<unsigned>((groups + kMaxRowBlocks - 1) / kMaxRowBlocks));
    ProfileScope ps("minhash_rows_kernel", stream);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(minhash_rows_kernel<T, K, TAIL>), grid, dim3(kThreads), 0, stream, v, seed, a, b, P, width, offsets, child,
                       per_wave);
  }
  ProfileScope ps("minhash_parts_kernel", stream);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(minhash_parts_kernel<T, K, TAIL>), dim3(static_cast<unsigned>(parts.waves / kWaves)), dim3(kThreads), 0, stream, parts,
                     seed, a, b, P, width, chunks, offsets, prefix, counter, child);
}

// How the parameters are shared out: chunks of K sets of 64 (every chunk hashes the windows again, and a lane without
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

// The launches of one minhash call: the row offsets of the result and the parts of every row, then the hashing kernels.
// prefix holds rows + 1 values, scan_tmp scan_temp_bytes(rows) bytes and one 64-bit counter behind them.
template <typename T>
void run_minhash(const ColView& v, T seed, const T* a, const T* b, int32_t P, int32_t width, int32_t* offsets, T* child, int64_t child_size,
                 uint32_t* prefix, uint64_t* scan_tmp, hipStream_t stream)
{
  int32_t const rows = v.size;
  RowParts const parts{v, device_cus() * 4 * minhash_waves<T>(), rows >= kManyRows ? kPartBytes : -1};
  auto* const counter = reinterpret_cast<unsigned long long*>(scan_tmp) + scan_temp_bytes(rows) / sizeof(uint64_t);
  if (rows <= kPlanRows) {
    int64_t const most    = std::max<int64_t>(child_size, rows + 1);
    unsigned const groups = static_cast<unsigned>(std::min<int64_t>((most + 4 * kScanThreads - 1) / (4 * kScanThreads), 1024));
    hipLaunchKernelGGL(HIP_KERNEL_NAME(minhash_plan_kernel<T>), dim3(1 + groups), dim3(kScanThreads), 0, stream, parts, P, offsets, prefix, counter, child,
                       child_size);
  } else {
    if (v.use_mask) {
      device_exclusive_scan(ValidTimesP{v, P}, static_cast<int64_t>(rows), offsets, scan_tmp, stream);
    } else {
      hipLaunchKernelGGL(uniform_offsets_kernel, dim3((rows + 1 + 255) / 256), dim3(256), 0, stream, offsets, rows, P);
    }
    device_exclusive_scan(parts, static_cast<int64_t>(rows), prefix, scan_tmp, stream);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(minhash_clear_kernel<T>), dim3((rows + kThreads - 1) / kThreads), dim3(kThreads), 0, stream, parts, P, offsets, counter,
                       child);
  }

  if (child_size > 0) {
    Sharing const sh = sharing_for(P);
    switch (sh.k * 2 + (sh.tail ? 1 : 0)) {
      case 10: launch_kernels<T, 5, false>(parts, seed, a, b, P, width, offsets, prefix, counter, child, stream); break;
      case 9: launch_kernels<T, 4, true>(parts, seed, a, b, P, width, offsets, prefix, counter, child, stream); break;
      case 8: launch_kernels<T, 4, false>(parts, seed, a, b, P, width, offsets, prefix, counter, child, stream); break;
      case 7: launch_kernels<T, 3, true>(parts, seed, a, b, P, width, offsets, prefix, counter, child, stream); break;
      case 6: launch_kernels<T, 3, false>(parts, seed, a, b, P, width, offsets, prefix, counter, child, stream); break;
      case 5: launch_kernels<T, 2, true>(parts, seed, a, b, P, width, offsets, prefix, counter, child, stream); break;
      case 4: launch_kernels<T, 2, false>(parts, seed, a, b, P, width, offsets, prefix, counter, child, stream); break;
      case 3: launch_kernels<T, 1, true>(parts, seed, a, b, P, width, offsets, prefix, counter, child, stream); break;
      default: launch_kernels<T, 1, false>(parts, seed, a, b, P, width, offsets, prefix, counter, child, stream); break;
    }
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
  size_t const temp_bytes[2] = {scan_temp_bytes(rows) + sizeof(uint64_t), static_cast<size_t>(rows + 1) * sizeof(uint32_t)};
  TempParts<2> const temp(mr, temp_bytes);
  if (!temp.ok()) {
    nvtext_amd_list_column_free(out, stream_, mr_);
    return fail(NVTEXT_AMD_ALLOC_FAILED, "temporary allocation failed");
  }
  run_minhash<T>(v, seed, a, b, P, width, out->offsets, static_cast<T*>(out->child), out->child_size, temp.part<uint32_t>(1),
                 temp.part<uint64_t>(0), stream);
  NVTEXT_HIP_TRY_OR(hipGetLastError(), nvtext_amd_list_column_free(out, stream_, mr_));
  return NVTEXT_AMD_SUCCESS;
}


// ------------------------------------------------------------------ minhash_ngrams / minhash64_ngrams
// LIST<STRING> rows: the hashed items are runs of consecutive list elements instead of character windows
// (cpp/src/text/minhash.cu:182-250); the permutation and the minimum are the ones above.
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
  __device__ __forceinline__ uint32_t u32(uint32_t i) const
  {
    uint32_t const o  = mis + i;
    uint32_t const j  = o >> 2;
    uint32_t const lo = w[j];
    uint32_t const hi = 4u * (j + 1u) < end ? w[j + 1] : 0u;
    return __builtin_amdgcn_alignbit(hi, lo, (o & 3u) * 8u);
  }
};

constexpr uint32_t kNgramStageBytes = 4096;                             // longest stretch of chars hashed out of LDS
constexpr uint32_t kNgramStageWords = (kNgramStageBytes + 16 + 32) / 4;  // + misalignment, + whole blocks and over-read of the hash tail

// One workgroup per (group of consecutive rows, parameter chunk), as in minhash_rows_kernel: a row of up to
// kNgramSoloPositions positions is done by one wavefront alone, 64 positions a trip (wavefront w takes the rows w, w + 4, .. of the group,
// `solo_per_wave` of them), and its minima go from the registers to the result; a row of more positions is shared by the
// four wavefronts, which take its positions 64 at a time in turn and combine through LDS, one such row after the other.
// A column of fewer than 131,072 rows keeps one row to a workgroup, every row shared by the four wavefronts
// (solo_per_wave 0): it needs its workgroups to fill the device and to even out its end (20,000 rows of 3,000 elements:
// four rows to a workgroup were 8 % slower).
constexpr int64_t kNgramSoloPositions = 2048;
template <typename T, int K>
__global__ void __launch_bounds__(kThreads) minhash_ngrams_kernel(ListView in, int32_t ngrams, T seed, const T* __restrict__ pa,
                                                                  const T* __restrict__ pb, int32_t P, const int32_t* __restrict__ out_offsets,
                                                                  T* __restrict__ out, int solo_per_wave)
{
  using H = HashTraits<T>;
  __shared__ alignas(16) T hashes[kWaves][2 * kWave];  // 64 hashes a trip, padded to the stride of the fold (at most 64 more)
  __shared__ T red[kWaves][K * kWave];
  // the chars of the elements a wavefront is hashing (32-bit hash only: measured 13 % faster there, 9 % slower for the
  // 64-bit hash, whose 16-byte steps cost more to assemble out of LDS than they save)
  constexpr bool kStageRuns = sizeof(T) == 4;
  __shared__ alignas(16) uint32_t run_bytes[kWaves][kStageRuns ? kNgramStageWords : 1];
  __shared__ uint32_t next_row;

  int const group_rows = solo_per_wave > 0 ? solo_per_wave * kWaves : 1;
  int64_t const r0     = (static_cast<int64_t>(blockIdx.z) * gridDim.x + blockIdx.x) * group_rows;  // groups along x, then z
  if (r0 >= in.size) return;
  int64_t const solo_positions = solo_per_wave > 0 ? kNgramSoloPositions : -1;
  int32_t const chunk_base     = blockIdx.y * (K * kWave);
  int32_t const in_chunk       = min(K * kWave, P - chunk_base);
  int const lane               = lane_id();
  int const wave               = threadIdx.x / kWave;
  T a[K], b[K], m[K];
  load_params<T, K>(pa, pb, P, chunk_base, lane, a, b, m);

  int const rows_here = static_cast<int>(min(static_cast<int64_t>(group_rows), in.size - r0));
  if (threadIdx.x == 0) next_row = 0;
  __syncthreads();
  // the short rows of the group first, each wavefront taking the next one whenever it is done with one; then, from
  // `together` = 0 on, the rows that all four do together, one after the other (see minhash_rows_kernel)
  int together = -1;
  for (;;) {
    int i;
    if (together < 0) {
      int t = 0;
      if (lane == 0) t = static_cast<int>(atomicAdd(&next_row, 1u));
      i = __builtin_amdgcn_readfirstlane(t);
      if (i >= rows_here) {
        together = 0;
        continue;
      }
    } else {
      if (together >= rows_here) break;
      i = together++;
    }
    bool const solo = together < 0;
    if (!in.valid(r0 + i)) continue;
    int64_t const first = in.off(r0 + i);
    int64_t const n     = in.off(r0 + i + 1) - first;
    // minhash.cu:311-314 with width = ngrams: the positions that the permutation looks at
    int64_t const positions = max(static_cast<int64_t>(1), n - ngrams + 1);
    if (solo != (positions <= solo_positions)) continue;
#pragma unroll
    for (int k = 0; k < K; ++k) m[k] = std::numeric_limits<T>::max();
    if (n > 0) {
      int64_t const trip = solo ? kWave : kWaves * kWave;
      for (int64_t base = solo ? 0 : static_cast<int64_t>(wave) * kWave; base < positions; base += trip) {
        int64_t const idx = base + lane;
        bool valid        = false;
        T hv              = 0;
        int64_t bo = 0, eo = 0;
        if (idx < positions && in.child.valid(first + idx)) {  // 213-216: a null element starts no run
          // 218-222: the run ends at element idx + ngrams, clamped to the row; a clamped run counts only at idx 0
          int64_t const next = min(idx + ngrams, n - 1);
          if (idx == 0 || next - idx >= ngrams) {
            // 224-229: the bytes from the start of element idx to the end of element next
            bo    = in.child.off(first + idx);
            eo    = in.child.off(first + next + 1);
            valid = true;
          }
        }
        // The runs of these 64 elements overlap and lie side by side in the chars: fetch that stretch once, with
        // coalesced loads, and hash out of LDS (the hash walks a run dword by dword, each step a dependent read).
        // A stretch too long for the buffer is hashed straight from memory.
        int64_t const span_begin = kStageRuns ? in.child.off(first + base) : 0;
        int64_t const span_end   = kStageRuns ? in.child.off(first + min(base + kWave + ngrams, n)) : 0;
        if (kStageRuns && span_end - span_begin <= static_cast<int64_t>(kNgramStageBytes)) {
          bool ascii;
          uint32_t const mis = stage_bytes(in.child.chars, span_begin, static_cast<uint32_t>(span_end - span_begin), run_bytes[wave], lane, &ascii);
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
          if (valid) {
            WordSrc const src{run_bytes[wave], mis + static_cast<uint32_t>(bo - span_begin)};
            hv = H::hash(src, static_cast<uint32_t>(eo - bo), seed);
          }
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
        } else if (valid) {
          AlignedSrc const src(in.child.chars + bo, static_cast<uint32_t>(eo - bo));
          hv = H::hash(src, static_cast<uint32_t>(eo - bo), seed);
        }
        if (valid) hv = hv < 1 ? T{1} : hv;  // 237
        uint64_t const vm = ballot64(valid);
        if (valid) hashes[wave][lanes_below(vm)] = hv;
        fold_hashes<T, K>(hashes[wave], static_cast<uint32_t>(__builtin_popcountll(vm)), a, b, m, lane);
      }
    }
    T* const dst = out + static_cast<int64_t>(out_offsets[r0 + i]) + chunk_base;
    if (solo) {
      // an empty row is zeros (minhash.cu:318); a row whose every run was skipped keeps the all-ones start value
#pragma unroll
      for (int k = 0; k < K; ++k) {
        int32_t const j = lane + kWave * k;
        if (j < in_chunk) dst[j] = n > 0 ? m[k] : T{0};
      }
    } else {
      __syncthreads();  // (the row before has been read out of red)
#pragma unroll
      for (int k = 0; k < K; ++k) red[wave][k * kWave + lane] = m[k];
      __syncthreads();
      for (int j = threadIdx.x; j < in_chunk; j += kThreads) {
        T v = red[0][j];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) v = min(v, red[w][j]);
        dst[j] = n > 0 ? v : T{0};
      }
    }
  }
}

struct ListValidTimesP {
  ListView in;
  int32_t P;
  __device__ uint64_t operator()(int64_t i) const { return in.valid(i) ? static_cast<uint64_t>(P) : 0; }
};

template <typename T, int K>
void launch_ngrams(const ListView& v, int32_t ngrams, T seed, const T* a, const T* b, int32_t P, const int32_t* offsets, T* child,
                   hipStream_t stream)
{
  int32_t const chunks    = (P + K * kWave - 1) / (K * kWave);
  int const solo_per_wave = v.size >= kManyRows ? rows_per_wave(v.size) : 0;
  int32_t const group     = solo_per_wave > 0 ? solo_per_wave * kWaves : 1;
  int32_t const groups    = (v.size + group - 1) / group;
  dim3 grid(static_cast<unsigned>(std::min(groups, kMaxRowBlocks)), static_cast<unsigned>(chunks),
            static_cast<unsigned>((groups + kMaxRowBlocks - 1) / kMaxRowBlocks));
  ProfileScope ps("minhash_ngrams_kernel", stream);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(minhash_ngrams_kernel<T, K>), grid, dim3(kThreads), 0, stream, v, ngrams, seed, a, b, P, offsets, child,
                     solo_per_wave);
}

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
  if (v.use_mask) {
    Temp scan_tmp(mr, scan_temp_bytes(rows));
    if (!scan_tmp.ok()) {
      nvtext_amd_list_column_free(out, stream_, mr_);
      return fail(NVTEXT_AMD_ALLOC_FAILED, "temporary allocation failed");
    }
    device_exclusive_scan(ListValidTimesP{v, P}, static_cast<int64_t>(rows), out->offsets, scan_tmp.as<uint64_t>(), stream);
  } else {
    hipLaunchKernelGGL(uniform_offsets_kernel, dim3((rows + 1 + 255) / 256), dim3(256), 0, stream, out->offsets, rows, P);
  }
  T* child = static_cast<T*>(out->child);
  if (out->child_size > 0) {
    if (P > 2 * kWave)
      launch_ngrams<T, 4>(v, ngrams, seed, a, b, P, out->offsets, child, stream);
    else if (P > kWave)
      launch_ngrams<T, 2>(v, ngrams, seed, a, b, P, out->offsets, child, stream);
    else
      launch_ngrams<T, 1>(v, ngrams, seed, a, b, P, out->offsets, child, stream);
  }
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
  uint64_t* const scan_tmp = reinterpret_cast<uint64_t*>(base + kScratchPrefixBytes);

  if (input->null_mask) launch_copy_bitmask(out_null_mask, input->null_mask, input->offset, rows, stream);
  ColView const v = make_view(*input);
  // every value of the scratch that the kernels read is written earlier in this same call: nothing to clear
  run_minhash<uint32_t>(v, seed, a, b, P, width, out_offsets, out_child, child_size, prefix, scan_tmp, stream);
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
