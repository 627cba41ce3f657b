// Shared host/device helpers for the gfx950 nvtext kernels: status reporting,
// stream-ordered temporaries, the device view of an Arrow strings column,
// wavefront (64-lane) DPP scans, workgroup scans and a device-wide exclusive scan.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <utility>
#include <vector>

#include "../../include/nvtext_amd.h"
#include "../../include/nvtext_amd_profile.h"

namespace nvtext_amd {

constexpr int kWave = 64;

// ------------------------------------------------------------------ status
void set_last_error(const char* msg);
nvtext_amd_status fail(nvtext_amd_status st, const char* msg);
// What every entry point does first.  (1) hipGetLastError keeps the last error of the calling thread until somebody
// reads it, whoever made the failing call (a device query of another library, long before): it is read away before the
// entry point's own launches, which are checked with the same call, so that it reports no error but its own.  (2) A
// named range around the call, as CUDF_FUNC_RANGE() puts an NVTX range around the reference's entry points
// (cpp/include/cudf/detail/nvtx/ranges.hpp; wordpiece_tokenize.cu:291,897, minhash.cu:699,724): rocprofv3
// --marker-trace shows it.  The marker library (rocTX) is looked up at first use and left alone when it is absent;
// the library does not link it.
struct EntryScope {
  explicit EntryScope(const char* name);
  ~EntryScope();
  EntryScope(const EntryScope&)            = delete;
  EntryScope& operator=(const EntryScope&) = delete;
};

#define NVTEXT_HIP_TRY(expr)                                                          \
  do {                                                                                \
    hipError_t _e = (expr);                                                           \
    if (_e != hipSuccess) {                                                           \
      std::string _m = std::string(#expr) + ": " + hipGetErrorString(_e);             \
      return ::nvtext_amd::fail(NVTEXT_AMD_DEVICE_ERROR, _m.c_str());                 \
    }                                                                                 \
  } while (0)

// The same once the result has buffers: `release` hands them back before the error is returned.
#define NVTEXT_HIP_TRY_OR(expr, release)                                              \
  do {                                                                                \
    hipError_t _e = (expr);                                                           \
    if (_e != hipSuccess) {                                                           \
      release;                                                                        \
      std::string _m = std::string(#expr) + ": " + hipGetErrorString(_e);             \
      return ::nvtext_amd::fail(NVTEXT_AMD_DEVICE_ERROR, _m.c_str());                 \
    }                                                                                 \
  } while (0)

// ------------------------------------------------------------------ kernel timing (benchmarks)
bool profiling_on();
void profile_mark_begin(const char* name, hipStream_t stream);
void profile_mark_end(hipStream_t stream);

// Brackets one kernel launch with HIP events when profiling is enabled.
struct ProfileScope {
  hipStream_t stream;
  bool on;
  ProfileScope(const char* name, hipStream_t s) : stream(s), on(profiling_on())
  {
    if (on) profile_mark_begin(name, stream);
  }
  ~ProfileScope()
  {
    if (on) profile_mark_end(stream);
  }
};

// ------------------------------------------------------------------ memory
// Stream-ordered allocation through the caller's allocator (or hipMallocAsync).
struct Mr {
  const nvtext_amd_allocator* a;
  hipStream_t stream;
  void* allocate(size_t bytes) const;
  void deallocate(void* p, size_t bytes) const;
};

// Device memory that an object keeps for as long as it lives.  With an allocator it comes from there and goes back
// there on the stream of creation (a copy of the struct is kept: its ctx and that stream must outlive the object,
// as a memory resource must outlive what it allocated); without one it is plain hipMalloc / hipFree.
struct DeviceStore {
  nvtext_amd_allocator alloc{};
  bool has_alloc     = false;
  hipStream_t stream = nullptr;
  std::vector<std::pair<void*, size_t>> held;

  void bind(const nvtext_amd_allocator* a, hipStream_t s)
  {
    has_alloc = a && a->allocate && a->deallocate;
    if (has_alloc) alloc = *a;
    stream = s;
  }
  void* allocate(size_t bytes)
  {
    void* p = nullptr;
    if (has_alloc) {
      p = alloc.allocate(alloc.ctx, bytes, stream);
    } else if (hipMalloc(&p, bytes) != hipSuccess) {
      p = nullptr;
    }
    if (p) held.emplace_back(p, bytes);
    return p;
  }
  template <typename T>
  bool allocate(T** out, size_t count)
  {
    *out = static_cast<T*>(allocate(count * sizeof(T)));
    return *out != nullptr;
  }
  void release()
  {
    for (auto const& h : held) {
      if (has_alloc)
        alloc.deallocate(alloc.ctx, h.first, h.second, stream);
      else
        (void)hipFree(h.first);
    }
    held.clear();
  }
  DeviceStore() = default;
  ~DeviceStore() { release(); }
  DeviceStore(const DeviceStore&)            = delete;
  DeviceStore& operator=(const DeviceStore&) = delete;
};

// Temporary released (stream-ordered) when it goes out of scope.
struct Temp {
  Mr mr;
  void* ptr   = nullptr;
  size_t size = 0;
  Temp(Mr m, size_t bytes) : mr(m), size(bytes)
  {
    if (bytes) ptr = mr.allocate(bytes);
  }
  ~Temp()
  {
    if (ptr) mr.deallocate(ptr, size);
  }
  Temp(const Temp&)            = delete;
  Temp& operator=(const Temp&) = delete;
  bool ok() const { return size == 0 || ptr != nullptr; }
  template <typename T>
  T* as() const
  {
    return static_cast<T*>(ptr);
  }
};

// Several temporaries in ONE allocation (a call to the caller's allocator can cost tens of microseconds: from Python
// it is a callback into the interpreter), each part 256-byte aligned.
template <int N>
struct TempParts {
  size_t at[N + 1];
  Temp whole;
  static size_t total(const size_t (&bytes)[N])
  {
    size_t sum = 0;
    for (int i = 0; i < N; ++i) sum += (bytes[i] + 255) & ~static_cast<size_t>(255);
    return sum;
  }
  // (wanted: false for no allocation at all)
  TempParts(Mr m, const size_t (&bytes)[N], bool wanted = true) : whole(m, wanted ? total(bytes) : 0)
  {
    at[0] = 0;
    for (int i = 0; i < N; ++i) at[i + 1] = at[i] + ((bytes[i] + 255) & ~static_cast<size_t>(255));
  }
  bool ok() const { return whole.ok(); }
  template <typename T>
  T* part(int i) const
  {
    return reinterpret_cast<T*>(static_cast<char*>(whole.ptr) + at[i]);
  }
};

inline size_t mask_alloc_bytes(int64_t bits)
{
  // libcudf pads bitmask allocations to 64 bytes (cpp/include/cudf/null_mask.hpp:56-57)
  size_t const bytes = static_cast<size_t>((bits + 7) / 8);
  return (bytes + 63) / 64 * 64;
}

// ------------------------------------------------------------------ column view on the device
struct ColView {
  const uint8_t* chars;
  const void* offsets;
  const uint32_t* mask;
  int32_t size;
  int32_t offset;
  int32_t is64;
  int32_t use_mask;  // 1 when validity must be consulted (mask present and null_count > 0)

  __device__ __forceinline__ int64_t off(int64_t i) const
  {
    return is64 ? static_cast<const int64_t*>(offsets)[i + offset]
                : static_cast<int64_t>(static_cast<const int32_t*>(offsets)[i + offset]);
  }
  __device__ __forceinline__ bool valid(int64_t i) const
  {
    if (!use_mask) return true;
    int64_t const b = i + offset;
    return (mask[b >> 5] >> (b & 31)) & 1u;
  }
};

inline ColView make_view(const nvtext_amd_strings_column& c)
{
  ColView v;
  v.chars    = reinterpret_cast<const uint8_t*>(c.chars);
  v.offsets  = c.offsets;
  v.mask     = c.null_mask;
  v.size     = c.size;
  v.offset   = c.offset;
  v.is64     = c.offsets_is_int64 ? 1 : 0;
  v.use_mask = (c.null_mask != nullptr && c.null_count > 0) ? 1 : 0;
  return v;
}

// ------------------------------------------------------------------ UTF-8
// cpp/include/cudf/strings/detail/utf8.hpp:23-27, 84-90
__device__ __forceinline__ bool is_utf8_continuation(uint32_t b) { return (b & 0xC0u) == 0x80u; }
__device__ __forceinline__ int bytes_in_utf8_byte(uint32_t b)
{
  return 1 + int((b & 0xF0u) == 0xF0u) + int((b & 0xE0u) == 0xE0u) + int((b & 0xC0u) == 0xC0u) -
         int((b & 0xC0u) == 0x80u);
}

// ------------------------------------------------------------------ wavefront primitives (wave64, DPP)
// Loads and stores for data that is touched once: the non-temporal hint lets the caches drop these lines
// first, so that tables which are probed again and again stay resident.
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 load_stream(const uint4* p)
{
  u32x4_t const v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void store_stream(uint4* p, uint4 v)
{
  u32x4_t w;
  w.x = v.x; w.y = v.y; w.z = v.z; w.w = v.w;
  __builtin_nontemporal_store(w, reinterpret_cast<u32x4_t*>(p));
}
__device__ __forceinline__ uint32_t load_stream(const uint32_t* p) { return __builtin_nontemporal_load(p); }
__device__ __forceinline__ void store_stream(uint32_t* p, uint32_t v) { __builtin_nontemporal_store(v, p); }
__device__ __forceinline__ void store_stream(int32_t* p, int32_t v) { __builtin_nontemporal_store(v, p); }

__device__ __forceinline__ int lane_id() { return static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u))); }

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_zero(uint32_t v)
{
  // lanes without a source (or masked-out rows) read 0
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, ROW_MASK, 0xf, false));
}

// Inclusive prefix sum across the 64 lanes: four row_shr steps inside each row of 16,
// then row_bcast:15 / row_bcast:31 carry the row totals forward.
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v)
{
  v += dpp_zero<0x111, 0xf>(v);  // row_shr:1
  v += dpp_zero<0x112, 0xf>(v);  // row_shr:2
  v += dpp_zero<0x114, 0xf>(v);  // row_shr:4
  v += dpp_zero<0x118, 0xf>(v);  // row_shr:8
  v += dpp_zero<0x142, 0xa>(v);  // row_bcast:15 -> rows 1,3
  v += dpp_zero<0x143, 0xc>(v);  // row_bcast:31 -> rows 2,3
  return v;
}

__device__ __forceinline__ uint64_t wave_inclusive_scan64(uint64_t v)
{
#define NVTEXT_DPP64(CTRL, RM)                                                                  \
  {                                                                                             \
    uint32_t lo = dpp_zero<CTRL, RM>(static_cast<uint32_t>(v));                                 \
    uint32_t hi = dpp_zero<CTRL, RM>(static_cast<uint32_t>(v >> 32));                           \
    v += (static_cast<uint64_t>(hi) << 32) | lo;                                                \
  }
  NVTEXT_DPP64(0x111, 0xf)
  NVTEXT_DPP64(0x112, 0xf)
  NVTEXT_DPP64(0x114, 0xf)
  NVTEXT_DPP64(0x118, 0xf)
  NVTEXT_DPP64(0x142, 0xa)
  NVTEXT_DPP64(0x143, 0xc)
#undef NVTEXT_DPP64
  return v;
}

__device__ __forceinline__ uint32_t wave_bcast(uint32_t v, int lane) { return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), lane)); }
__device__ __forceinline__ uint64_t wave_bcast64(uint64_t v, int lane)
{
  uint32_t lo = wave_bcast(static_cast<uint32_t>(v), lane);
  uint32_t hi = wave_bcast(static_cast<uint32_t>(v >> 32), lane);
  return (static_cast<uint64_t>(hi) << 32) | lo;
}

__device__ __forceinline__ uint64_t ballot64(bool p) { return __builtin_amdgcn_ballot_w64(p); }
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask)
{
  return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u));
}

// What the lanes of a wavefront have written to its part of LDS is there for all of them.
__device__ __forceinline__ void wave_lds_fence()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// (written out, the compiler shares its inner minimum with a three-way minimum next to it, which then takes two instructions)
__device__ __forceinline__ uint32_t median(uint32_t a, uint32_t b, uint32_t c)
{
  uint32_t m;
  asm("v_med3_u32 %0, %1, %2, %3" : "=v"(m) : "v"(a), "v"(b), "v"(c));
  return m;
}

// Workgroup exclusive scan of one uint32 per thread.  `lds` needs (blockDim/64 + 1) words.
// Returns the exclusive prefix; *total receives the workgroup sum (same value on every thread).
template <int THREADS>
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* lds, uint32_t* total)
{
  constexpr int W  = THREADS / kWave;
  int const lane   = lane_id();
  int const wave   = threadIdx.x / kWave;
  uint32_t const i = wave_inclusive_scan(v);
  __syncthreads();  // protect lds reuse between calls
  if (lane == kWave - 1) lds[wave] = i;
  __syncthreads();
  uint32_t base = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    uint32_t const t = lds[w];
    if (w < wave) base += t;
    sum += t;
  }
  *total = sum;
  return base + i - v;
}

// Workgroup barrier that orders LDS traffic only: global loads issued before it stay in flight (a __syncthreads()
// waits for them).  For kernels whose lanes exchange data through LDS alone.
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// block_exclusive_scan with lds_barrier() in place of __syncthreads().
template <int THREADS>
__device__ __forceinline__ uint32_t block_exclusive_scan_lds(uint32_t v, uint32_t* lds, uint32_t* total)
{
  constexpr int W  = THREADS / kWave;
  int const lane   = lane_id();
  int const wave   = threadIdx.x / kWave;
  uint32_t const i = wave_inclusive_scan(v);
  lds_barrier();  // protect lds reuse between calls
  if (lane == kWave - 1) lds[wave] = i;
  lds_barrier();
  uint32_t base = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    uint32_t const t = lds[w];
    if (w < wave) base += t;
    sum += t;
  }
  *total = sum;
  return base + i - v;
}

template <int THREADS>
__device__ __forceinline__ uint64_t block_exclusive_scan64(uint64_t v, uint64_t* lds, uint64_t* total)
{
  constexpr int W  = THREADS / kWave;
  int const lane   = lane_id();
  int const wave   = threadIdx.x / kWave;
  uint64_t const i = wave_inclusive_scan64(v);
  __syncthreads();
  if (lane == kWave - 1) lds[wave] = i;
  __syncthreads();
  uint64_t base = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    uint64_t const t = lds[w];
    if (w < wave) base += t;
    sum += t;
  }
  *total = sum;
  return base + i - v;
}

// ------------------------------------------------------------------ device-wide exclusive scan
// out[i] = sum_{j<i} f(j) for i in [0, n]  (n+1 entries; out[n] is the total), and tell(total) by one thread as soon as the total
// is known.
// Two launches: the sums of the tiles; then every workgroup adds up the sums before its own, and the first all of them.  (With a
// launch of its own for the scan of the sums, and another to tell the host, calls of 26 to 770 MB took 4 to 6 us more.)
// Three where there are more than kScanDirect tiles, one for a few thousand values.
constexpr int kScanThreads    = 256;
constexpr int kScanItems      = 8;
constexpr int kScanTile       = kScanThreads * kScanItems;
constexpr int64_t kScanDirect = 1024;

struct TellNobody {
  __device__ void operator()(uint64_t) const {}
};

template <typename F>
__global__ void __launch_bounds__(kScanThreads) scan_tile_sums_kernel(F f, int64_t n, uint64_t* tile_sums)
{
  __shared__ uint64_t lds[kScanThreads / kWave + 1];
  int64_t const base = static_cast<int64_t>(blockIdx.x) * kScanTile + static_cast<int64_t>(threadIdx.x) * kScanItems;
  uint64_t s         = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int64_t const i = base + k;
    if (i < n) s += f(i);
  }
  uint64_t total;
  block_exclusive_scan64<kScanThreads>(s, lds, &total);
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

// exclusive scan of tile_sums in place; tile_sums[ntiles] = grand total
template <typename Tell>
__global__ void __launch_bounds__(kScanThreads) scan_tile_offsets_kernel(uint64_t* tile_sums, int64_t ntiles, Tell tell)
{
  __shared__ uint64_t lds[kScanThreads / kWave + 1];
  uint64_t carry = 0;
  for (int64_t base = 0; base < ntiles; base += kScanThreads) {
    int64_t const i  = base + threadIdx.x;
    uint64_t const v = (i < ntiles) ? tile_sums[i] : 0;
    uint64_t total;
    uint64_t const ex = block_exclusive_scan64<kScanThreads>(v, lds, &total);
    if (i < ntiles) tile_sums[i] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) {
    tile_sums[ntiles] = carry;
    tell(carry);
  }
}

// SUMS: `tiles` holds the sums of the tiles as they are, and the first workgroup adds all of them up (tiles[number of tiles] = the
// grand total); else what comes before each.
template <bool SUMS, typename F, typename OutT, typename Tell>
__global__ void __launch_bounds__(kScanThreads) scan_apply_kernel(F f, int64_t n, uint64_t* tiles, OutT* out, Tell tell)
{
  __shared__ uint64_t lds[kScanThreads / kWave + 1];
  int64_t const base = static_cast<int64_t>(blockIdx.x) * kScanTile + static_cast<int64_t>(threadIdx.x) * kScanItems;
  uint64_t vals[kScanItems];
  uint64_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int64_t const i = base + k;
    vals[k]         = (i < n) ? static_cast<uint64_t>(f(i)) : 0;
    s += vals[k];
  }
  uint64_t total, before = 0;
  if constexpr (SUMS) {
    uint32_t const mine = blockIdx.x == 0 ? gridDim.x : blockIdx.x;  // (the first workgroup needs none before its own)
    uint64_t part       = 0;
#pragma unroll
    for (uint32_t k = 0; k < kScanDirect / kScanThreads; ++k) {
      uint32_t const i = k * kScanThreads + threadIdx.x;
      if (i < mine) part += tiles[i];
    }
    block_exclusive_scan64<kScanThreads>(part, lds, &before);
    if (blockIdx.x == 0) {
      if (threadIdx.x == 0) {
        tiles[gridDim.x] = before;
        tell(before);
      }
      before = 0;
    }
  } else {
    before = tiles[blockIdx.x];
  }
  uint64_t run = block_exclusive_scan64<kScanThreads>(s, lds, &total) + before;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int64_t const i = base + k;
    if (i < n) out[i] = static_cast<OutT>(run);
    run += vals[k];
    if (i == n - 1) out[n] = static_cast<OutT>(run);
  }
}

// The whole scan by one workgroup, for the few thousand values of a small call: one launch.
// tile_sums[tiles] receives the grand total, as the others leave it.
constexpr int64_t kScanSmallTiles = 4;
template <typename F, typename OutT, typename Tell>
__global__ void __launch_bounds__(kScanThreads) scan_small_kernel(F f, int64_t n, uint64_t* total_out, OutT* out, Tell tell)
{
  __shared__ uint64_t lds[kScanThreads / kWave + 1];
  uint64_t carry = 0;
  for (int64_t tile = 0; tile * kScanTile < n; ++tile) {
    int64_t const base = tile * kScanTile + static_cast<int64_t>(threadIdx.x) * kScanItems;
    uint64_t vals[kScanItems];
    uint64_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      int64_t const i = base + k;
      vals[k]         = (i < n) ? static_cast<uint64_t>(f(i)) : 0;
      s += vals[k];
    }
    uint64_t total;
    uint64_t run = block_exclusive_scan64<kScanThreads>(s, lds, &total) + carry;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      int64_t const i = base + k;
      if (i < n) out[i] = static_cast<OutT>(run);
      run += vals[k];
    }
    carry += total;
  }
  if (threadIdx.x == 0) {
    out[n]     = static_cast<OutT>(carry);
    *total_out = carry;
    tell(carry);
  }
}

inline int64_t scan_tiles(int64_t n) { return (n + kScanTile - 1) / kScanTile; }
inline size_t scan_temp_bytes(int64_t n) { return static_cast<size_t>(scan_tiles(n) + 1) * sizeof(uint64_t); }

// `temp` holds scan_temp_bytes(n) bytes; temp[ntiles] receives the grand total (uint64).
// n must be > 0.
template <typename F, typename OutT, typename Tell>
void device_exclusive_scan(F f, int64_t n, OutT* out, uint64_t* temp, hipStream_t stream, Tell tell)
{
  int64_t const tiles = scan_tiles(n);
  dim3 const grid(static_cast<unsigned>(tiles));
  if (tiles <= kScanSmallTiles) {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(scan_small_kernel<F, OutT, Tell>), dim3(1), dim3(kScanThreads), 0, stream, f, n, temp + tiles, out, tell);
    return;
  }
  hipLaunchKernelGGL(HIP_KERNEL_NAME(scan_tile_sums_kernel<F>), grid, dim3(kScanThreads), 0, stream, f, n, temp);
  if (tiles <= kScanDirect) {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(scan_apply_kernel<true, F, OutT, Tell>), grid, dim3(kScanThreads), 0, stream, f, n, temp, out, tell);
    return;
  }
  hipLaunchKernelGGL(HIP_KERNEL_NAME(scan_tile_offsets_kernel<Tell>), dim3(1), dim3(kScanThreads), 0, stream, temp, tiles, tell);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(scan_apply_kernel<false, F, OutT, TellNobody>), grid, dim3(kScanThreads), 0, stream, f, n, temp, out, TellNobody{});
}

// Compute units of the current device (read once per device).
int device_cus();

// ------------------------------------------------------------------ scalars for the host
// A little pinned host memory that kernels write and the host reads (a copy of a few bytes into ordinary host memory
// goes through a staging buffer and costs ten microseconds and more): eight 64-bit words, and a word in a cache line of its
// own that says what has been written.  One buffer per host thread, allocated at the thread's first call and kept until the
// process ends; nullptr when the allocation failed (the callers then copy).
constexpr size_t kHostPostedWord  = 16;  // (in 64-bit words)
constexpr size_t kHostScalarBytes = (kHostPostedWord + 16) * sizeof(uint64_t);
uint64_t* host_scalars();

// Word from a kernel that what it (and the kernels before it on its stream) wrote to the pinned words is there.  The host
// looks for it itself: it has the numbers some seven microseconds earlier than by waiting for the stream, and need not wait
// for kernels behind this one.
struct HostPost {
  uint64_t* posted;
  uint64_t ticket;
  // by one thread, after what it is about has been written: by this thread, or before a barrier with a fence of its own
  // (__threadfence_system) by the thread that wrote
  __device__ __forceinline__ void send() const
  {
    __threadfence_system();
    __hip_atomic_store(posted, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
};
HostPost new_post();  // (only where host_scalars() gives memory)
// Returns when it has been sent, or with the error that keeps it from being sent.
hipError_t wait_for_post(HostPost const& post, hipStream_t stream);

// By LANES neighbouring lanes (`member` is a lane's number among them; the whole wavefront comes along): the first of [lo, hi) that is not
// before(i), or hi; all of them look at once, an even distance apart, and a LANES-th of what was left remains.
template <int LANES, typename Before>
__device__ __forceinline__ uint32_t search_by_lanes(uint32_t lo, uint32_t hi, uint32_t member, Before const& before)
{
  while (ballot64(lo < hi) != 0) {
    auto const place     = [length = hi - lo, lo](uint32_t i) { return lo + static_cast<uint32_t>(static_cast<uint64_t>(length) * i / LANES); };
    bool const yes       = lo < hi && before(place(member));
    uint32_t const n     = __builtin_popcount(static_cast<uint32_t>(ballot64(yes) >> (lane_id() & ~(LANES - 1))) & ((1u << LANES) - 1u));  // the first n
    uint32_t const first = n > 0 ? place(n - 1u) + 1u : lo, last = n < LANES ? place(n) : hi;
    if (lo < hi) {
      lo = first;
      hi = last;
    }
  }
  return lo;
}

// What the workgroups of one launch add up between them, so that the last to arrive knows the sum and need not be another
// kernel: `sum` counts them in its upper bits.  Zeros between launches, which the last workgroup sees to.  Every host thread has
// one of its own on every device (device memory of the library, no allocation), given back when the thread ends.  For entry points
// that wait until the last workgroup has spoken: the thread's next call, on whatever stream, then finds zeros.
struct alignas(128) Arrivals {
  unsigned long long sum;
  uint32_t notes;
  alignas(128) uint32_t words[16];  // counters of the launch's own
};
constexpr int kMostArrivals = 1024;
Arrivals* thread_arrivals();  // (nullptr: as many threads as that have one)
// After a failure it may hold anything: no thread gets it any more, and this one another at its next call.
void forsake_thread_arrivals();
void launch_fill_u32(uint32_t* dst, uint32_t value, int64_t count, hipStream_t stream);
// What a call adds up in: the thread's, or, where there is none for it, memory of its own, zeroed first (a launch more).
class CallArrivals {
  Arrivals* const threads_;
  Temp const own_;

 public:
  CallArrivals(Mr mr, bool wanted) : threads_(wanted ? thread_arrivals() : nullptr), own_(mr, wanted && !threads_ ? sizeof(Arrivals) : 0)
  {
    if (own_.ptr) launch_fill_u32(own_.as<uint32_t>(), 0u, sizeof(Arrivals) / sizeof(uint32_t), mr.stream);
  }
  Arrivals* get() const { return threads_ ? threads_ : own_.as<Arrivals>(); }  // (nullptr: not wanted, or no memory)
  void failed() const
  {
    if (threads_) forsake_thread_arrivals();
  }
};

// dst[0] = offsets[first_index], dst[1] = offsets[last_index] (offsets of 32 or 64 bits)
void launch_read_two_offsets(const void* offsets, int is64, int64_t first_index, int64_t last_index, uint64_t* dst, HostPost post,
                             hipStream_t stream);

// ------------------------------------------------------------------ bitmask copy
// dst bit i = src bit (i + begin_bit); bits past `bits` are cleared
// (cpp/src/bitmask/null_mask.cu:332-347).
void launch_copy_bitmask(uint32_t* dst, const uint32_t* src, int32_t begin_bit, int32_t bits, hipStream_t stream);


}  // namespace nvtext_amd
