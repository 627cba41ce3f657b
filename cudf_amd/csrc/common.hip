// Host-side plumbing shared by the entry points: status text, allocator adaptor,
// bitmask copy, fills and the small
// C-ABI utilities (version, last error, result release).
#include "common.cuh"

#include <atomic>
#include <chrono>
#include <cstring>
#include <mutex>
#include <vector>

#include <dlfcn.h>

namespace nvtext_amd {

namespace {
thread_local std::string g_last_error;

struct ProfileRecord {
  const char* name;
  hipEvent_t begin;
  hipEvent_t end;
};
bool g_profile_on   = false;
bool g_profile_open = false;  // the last profile_mark_begin made a record
std::vector<ProfileRecord> g_profile;
}  // namespace

bool profiling_on() { return g_profile_on; }

void profile_mark_begin(const char* name, hipStream_t stream)
{
  ProfileRecord r{name, nullptr, nullptr};
  g_profile_open = false;
  if (hipEventCreate(&r.begin) != hipSuccess) return;
  if (hipEventCreate(&r.end) != hipSuccess) {
    (void)hipEventDestroy(r.begin);
    return;
  }
  (void)hipEventRecord(r.begin, stream);
  g_profile.push_back(r);
  g_profile_open = true;
}

void profile_mark_end(hipStream_t stream)
{
  // only the record that the matching begin made: a begin that failed leaves nothing to close
  if (g_profile_open) (void)hipEventRecord(g_profile.back().end, stream);
  g_profile_open = false;
}

namespace {
using RangePushFn = int (*)(const char*);
using RangePopFn  = int (*)();
RangePushFn g_range_push = nullptr;
RangePopFn g_range_pop   = nullptr;
std::once_flag g_range_once;
void find_marker_library()
{
  // rocprofv3 listens to the first; the second is the older tracer's
  for (const char* lib : {"librocprofiler-sdk-roctx.so.1", "libroctx64.so.4"}) {
    void* const h = dlopen(lib, RTLD_NOW | RTLD_LOCAL);
    if (!h) continue;
    auto const push = reinterpret_cast<RangePushFn>(dlsym(h, "roctxRangePushA"));
    auto const pop  = reinterpret_cast<RangePopFn>(dlsym(h, "roctxRangePop"));
    if (push && pop) {
      g_range_push = push;
      g_range_pop  = pop;
      return;
    }
  }
}
}  // namespace

EntryScope::EntryScope(const char* name)
{
  (void)hipGetLastError();
  std::call_once(g_range_once, find_marker_library);
  if (g_range_push) (void)g_range_push(name);
}

EntryScope::~EntryScope()
{
  if (g_range_pop) (void)g_range_pop();
}

void set_last_error(const char* msg) { g_last_error = msg ? msg : ""; }

nvtext_amd_status fail(nvtext_amd_status st, const char* msg)
{
  set_last_error(msg);
  return st;
}

void* Mr::allocate(size_t bytes) const
{
  if (bytes == 0) return nullptr;
  if (a && a->allocate) return a->allocate(a->ctx, bytes, stream);
  void* p = nullptr;
  if (hipMallocAsync(&p, bytes, stream) != hipSuccess) return nullptr;
  return p;
}

void Mr::deallocate(void* p, size_t bytes) const
{
  if (!p) return;
  if (a && a->deallocate) {
    a->deallocate(a->ctx, p, bytes, stream);
    return;
  }
  (void)hipFreeAsync(p, stream);
}

namespace {
__global__ void copy_bitmask_kernel(uint32_t* dst, const uint32_t* src, int32_t begin_bit, int32_t bits, int32_t words)
{
  int32_t const w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= words) return;
  int64_t const first = static_cast<int64_t>(begin_bit) + static_cast<int64_t>(w) * 32;
  int64_t const sw    = first >> 5;
  int const sh        = static_cast<int>(first & 31);
  int64_t const last_src_word = (static_cast<int64_t>(begin_bit) + bits - 1) >> 5;
  uint32_t v = src[sw] >> sh;
  if (sh != 0 && sw + 1 <= last_src_word) v |= src[sw + 1] << (32 - sh);
  int32_t const remaining = bits - w * 32;
  if (remaining < 32) v &= (1u << remaining) - 1u;
  dst[w] = v;
}

__global__ void fill_u32_kernel(uint32_t* dst, uint32_t value, int64_t count)
{
  int64_t const stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += stride) dst[i] = value;
}
}  // namespace

namespace {
__global__ void read_two_offsets_kernel(const void* offsets, int is64, int64_t first_index, int64_t last_index, uint64_t* dst, HostPost post)
{
  for (int k = 0; k < 2; ++k) {
    int64_t const i = k == 0 ? first_index : last_index;
    dst[k] = static_cast<uint64_t>(is64 ? static_cast<const int64_t*>(offsets)[i] : static_cast<int64_t>(static_cast<const int32_t*>(offsets)[i]));
  }
  post.send();
}
}  // namespace

int device_cus()
{
  constexpr int kMost = 64;
  static std::atomic<int> known[kMost] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMost) return 256;
  int cus = known[device].load(std::memory_order_relaxed);
  if (cus == 0) {
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0) cus = 256;
    known[device].store(cus, std::memory_order_relaxed);
  }
  return cus;
}

uint64_t* host_scalars()
{
  struct Slot {
    uint64_t* p = nullptr;
    bool tried  = false;
  };
  thread_local Slot slot;
  if (!slot.tried) {
    slot.tried = true;
    void* p    = nullptr;
    // portable: usable whichever device the thread has current at a later call
    // coherent: what a running kernel writes can be seen
    if (hipHostMalloc(&p, kHostScalarBytes, hipHostMallocPortable | hipHostMallocCoherent) == hipSuccess) {
      slot.p                  = static_cast<uint64_t*>(p);
      slot.p[kHostPostedWord] = 0;
    } else {
      (void)hipGetLastError();
    }
  }
  return slot.p;
}

namespace {
__device__ Arrivals g_arrivals[kMostArrivals];  // zeros when the library is loaded

// The numbers that no thread has.  (Never destroyed: threads end after the objects of the library do.)
struct FreeArrivals {
  std::mutex lock;
  std::vector<int> numbers;
  std::vector<int> held;  // (see nvtext_amd_profile_hold_arrivals)
  FreeArrivals()
  {
    for (int i = kMostArrivals; i-- > 0;) numbers.push_back(i);
  }
};
FreeArrivals& free_arrivals()
{
  static FreeArrivals* const all = new FreeArrivals;
  return *all;
}
struct ThreadArrivals {
  static constexpr int kDevices = 64;
  int number                    = -1;  // (none)
  Arrivals* first[kDevices]     = {};  // of the device's array
  bool take()
  {
    if (number >= 0) return true;
    FreeArrivals& all = free_arrivals();
    std::lock_guard<std::mutex> const guard(all.lock);
    if (all.numbers.empty()) return false;
    number = all.numbers.back();
    all.numbers.pop_back();
    return true;
  }
  ~ThreadArrivals()
  {
    if (number < 0) return;
    FreeArrivals& all = free_arrivals();
    std::lock_guard<std::mutex> const guard(all.lock);
    all.numbers.push_back(number);
  }
};
ThreadArrivals& of_this_thread()
{
  thread_local ThreadArrivals mine;
  return mine;
}
}  // namespace

Arrivals* thread_arrivals()
{
  ThreadArrivals& mine = of_this_thread();
  int device           = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= ThreadArrivals::kDevices || !mine.take()) return nullptr;
  if (!mine.first[device]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(g_arrivals)) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    mine.first[device] = static_cast<Arrivals*>(p);
  }
  return mine.first[device] + mine.number;
}

void forsake_thread_arrivals() { of_this_thread().number = -1; }

HostPost new_post()
{
  thread_local uint64_t tickets = 0;
  return HostPost{host_scalars() + kHostPostedWord, ++tickets};
}

hipError_t wait_for_post(HostPost const& post, hipStream_t stream)
{
  auto const sent = [&] { return __atomic_load_n(post.posted, __ATOMIC_ACQUIRE) == post.ticket; };
  auto asked = std::chrono::steady_clock::now();
  for (;;) {
    for (int look = 0; look < 64; ++look) {
      if (sent()) return hipSuccess;
      __builtin_ia32_pause();
    }
    // now and then the stream is asked: a kernel that failed sends nothing (seldom, because asking puts a marker on the
    // stream: asked every 30 us, calls of 55 us took 67)
    auto const now = std::chrono::steady_clock::now();
    if (now - asked < std::chrono::milliseconds(2)) continue;
    asked = now;
    hipError_t const e = hipStreamQuery(stream);
    if (e == hipErrorNotReady) {
      (void)hipGetLastError();
      continue;
    }
    if (e != hipSuccess) return e;
    return sent() ? hipSuccess : hipErrorUnknown;
  }
}

void launch_read_two_offsets(const void* offsets, int is64, int64_t first_index, int64_t last_index, uint64_t* dst, HostPost post, hipStream_t stream)
{
  hipLaunchKernelGGL(read_two_offsets_kernel, dim3(1), dim3(1), 0, stream, offsets, is64, first_index, last_index, dst, post);
}

void launch_copy_bitmask(uint32_t* dst, const uint32_t* src, int32_t begin_bit, int32_t bits, hipStream_t stream)
{
  int32_t const words = (bits + 31) / 32;
  if (words == 0) return;
  hipLaunchKernelGGL(copy_bitmask_kernel, dim3((words + 255) / 256), dim3(256), 0, stream, dst, src, begin_bit, bits, words);
}

void launch_fill_u32(uint32_t* dst, uint32_t value, int64_t count, hipStream_t stream)
{
  if (count <= 0) return;
  int64_t blocks = (count + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(fill_u32_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, dst, value, count);
}

}  // namespace nvtext_amd

extern "C" {

int32_t nvtext_amd_version(void) { return 100; }

void nvtext_amd_profile_enable(int32_t on)
{
  nvtext_amd::g_profile_on = on != 0;
}

int32_t nvtext_amd_profile_read(const char** names, float* milliseconds, int32_t capacity)
{
  int32_t n = 0;
  for (auto& r : nvtext_amd::g_profile) {
    float ms = 0.f;
    if (r.begin && r.end && hipEventSynchronize(r.end) == hipSuccess && hipEventElapsedTime(&ms, r.begin, r.end) == hipSuccess &&
        n < capacity) {
      names[n]        = r.name;
      milliseconds[n] = ms;
      ++n;
    }
    if (r.begin) (void)hipEventDestroy(r.begin);
    if (r.end) (void)hipEventDestroy(r.end);
  }
  nvtext_amd::g_profile.clear();
  return n;
}

int32_t nvtext_amd_profile_hold_arrivals(int32_t count)
{
  nvtext_amd::forsake_thread_arrivals();
  auto& all = nvtext_amd::free_arrivals();
  std::lock_guard<std::mutex> const guard(all.lock);
  auto const move = [](std::vector<int>& from, std::vector<int>& to) {
    to.push_back(from.back());
    from.pop_back();
  };
  while (static_cast<int32_t>(all.held.size()) < count && !all.numbers.empty()) move(all.numbers, all.held);
  while (static_cast<int32_t>(all.held.size()) > count && !all.held.empty()) move(all.held, all.numbers);
  return static_cast<int32_t>(all.numbers.size());
}

const char* nvtext_amd_last_error(void) { return nvtext_amd::g_last_error.c_str(); }

void nvtext_amd_list_column_free(nvtext_amd_list_column* col, void* stream, const nvtext_amd_allocator* mr)
{
  if (!col) return;
  nvtext_amd::Mr m{mr, static_cast<hipStream_t>(stream)};
  m.deallocate(col->offsets, col->offsets_bytes);
  m.deallocate(col->child, col->child_bytes);
  m.deallocate(col->null_mask, col->null_mask_bytes);
  std::memset(col, 0, sizeof(*col));
}

}  // extern "C"
