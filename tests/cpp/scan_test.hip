// device_exclusive_scan() of the library's headers over values in memory, for test_scan_gpu.py.
#include "../../cudf_amd/csrc/common.cuh"

namespace {
struct Values {
  const uint32_t* at;
  __device__ uint64_t operator()(int64_t i) const { return at[i]; }
};
struct TellTotal {
  uint64_t* at;
  __device__ void operator()(uint64_t total) const { *at = total; }
};
}  // namespace

// out: n + 1 entries; temp: scan_test_temp_bytes(n); total: what the scan tells, temp_total: what it leaves behind the sums.
extern "C" size_t scan_test_temp_bytes(int64_t n) { return nvtext_amd::scan_temp_bytes(n); }
extern "C" int64_t scan_test_lines(int which)
{
  int64_t const lines[3] = {nvtext_amd::kScanTile, nvtext_amd::kScanSmallTiles, nvtext_amd::kScanDirect};
  return lines[which];
}
extern "C" int scan_test(const uint32_t* values, int64_t n, int64_t* out, uint64_t* temp, uint64_t* total, void* stream)
{
  nvtext_amd::device_exclusive_scan(Values{values}, n, out, temp, static_cast<hipStream_t>(stream), TellTotal{total});
  return static_cast<int>(hipGetLastError());
}
