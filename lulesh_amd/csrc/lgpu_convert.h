// lgpu_convert.h -- fields between the caller's FP64 arrays and the device, by
// kernels: small ones, and the fields that the mixed form stores in FP32 (p,
// q, ss and the Q gradients).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

namespace lgpu {

// Whether a field of n values in the caller's array `host` is converted on the
// device instead of the host.  Twice the bytes then cross the link, which pinned
// memory takes at 55 GB/s, but other memory only at the rate of the copy into the
// runtime's buffers.  Host / device, us: pinned, upload 125,000 values 36.1 / 39.0,
// 166,375 47.0 / 45.0, 1,000,000 249 / 166, download 103,823 37.4 / 35.2, 1,000,000
// 362 / 167; not pinned, upload 216,000 62.4 / 85.0, 1,000,000 261 / 249, 2,744,000
// 832 / 623, download 216,000 74.3 / 121, 1,000,000 376 / 500, 7,077,888 3,797 / 3,695.
bool converts_on_device(const void *host, int64_t n, bool upload);

// dst[i] = (float)src[i] and dst[i] = src[i] on stream st.  Enqueue only.
hipError_t launch_narrow(const double *src, float *dst, int64_t n, hipStream_t st);
hipError_t launch_widen(const float *src, double *dst, int64_t n, hipStream_t st);

// Small fields are copied by a kernel between pinned memory and the device,
// waited for by its counts: hipMemcpy takes 12 us below 16 KiB and another path
// above.  Upload, hipMemcpy / so, us: 512 values 12.4 / 8.5, 1,728 12.6 / 9.8, 4,096
// 9.8 / 10.7.  hipMemcpy has to wait for the stream, 9 us after a kernel, so a
// context copies all of its fields one way (copies_by_kernel).
constexpr int kSmallProblem = 4096, kSmallMembers = 16384; // largest fields
constexpr int kSmallWave = 128; // values per wave
constexpr size_t small_copy_bytes(int values) // pinned memory; values a multiple of kSmallWave
{
   return sizeof(double) * (size_t)values + sizeof(uint32_t) * (size_t)(values / kSmallWave);
}

// Whether the kernel takes less time over the 6 node and 5 element fields of a
// state, for each problem's nodes and elements; those above `limit` go by
// hipMemcpy in any case.  fp32: 3 of the element fields are FP32 on the device.
inline bool copies_by_kernel(const std::vector<int32_t> &nodes, const std::vector<int32_t> &elems, int limit,
                             bool fp32)
{
   double kernel = 0., memcpy = 0.; // us
   auto add = [&](double fields, double n, double bytes) {
      const double m = n * bytes <= 16384. ? 12.4 : 8.7 + 0.00025 * n;
      const double k = 7.6 + 0.0008 * std::min(n, 4096.) + 0.0005 * std::max(n - 4096., 0.);
      memcpy += fields * m;
      kernel += fields * (n <= limit ? k : m + 9.0);
   };
   for (int32_t n : nodes) add(6., n, 8.);
   for (int32_t n : elems) {
      add(2., n, 8.);
      add(3., n, fp32 ? 4. : 8.);
   }
   return kernel < memcpy;
}

// The copies of one context: not for two threads at a time, as the context.
struct SmallCopy {
   int limit = 0; // largest field, 0 where hipMemcpy copies all
   double *buffer = nullptr;
   uint32_t *counts = nullptr;
   uint32_t seq = 0;
   void init(void *pinned); // small_copy_bytes(limit), aligned to 16
   bool takes(size_t n) const { return n <= (size_t)limit; }
   // Complete on return; after the stream's earlier work.  fp32: on the device.
   hipError_t upload(const double *host, void *device, bool fp32, int n, hipStream_t st);
   hipError_t download(void *device, double *host, bool fp32, int n, hipStream_t st);

 private:
   hipError_t wait(int n, hipStream_t st);
};

} // namespace lgpu
