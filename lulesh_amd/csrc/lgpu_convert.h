// lgpu_convert.h -- fields between the caller's FP64 arrays and the device, by
// kernels: small ones, and the fields that the mixed form stores in FP32 (p,
// q, ss and the Q gradients).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lgpu {

// Fields of up to this many values are converted on the host, where a launch
// and its synchronisation cost more than the loop: upload on the host / on the
// device, 27,000 values 14.8 / 25.4 us, 91,125 34.5 / 34.4, 250,047 69.6 / 56.7.
constexpr int64_t kConvertOnHost = 98304;

// dst[i] = (float)src[i] and dst[i] = src[i] on stream st.  Enqueue only.
hipError_t launch_narrow(const double *src, float *dst, int64_t n, hipStream_t st);
hipError_t launch_widen(const float *src, double *dst, int64_t n, hipStream_t st);

// Small fields are copied by a kernel between pinned memory and the device,
// waited for by its counts, where hipMemcpy would take less than 16 KiB: it has
// another path above that.  Upload and download, hipMemcpy / so, FP64: 512
// values 12.4 and 12.6 / 8.5 and 8.1 us, 1,728 12.6 and 13.0 / 9.8 and 9.4, 4,096
// 9.8 and 9.9 / 10.7 and 10.7; FP32 on the device: 4,096 12.9 and 13.4 / 11.7 and
// 10.8, 8,000 10.4 and 10.8 / 12.8 and 12.6.  An ensemble with such a member
// copies up to kMemberCopy values so, since hipMemcpy has to wait for the
// stream, 8 us after a kernel: 11 fields of 24 members of 5..24, 3.50 and 3.70
// ms / 2.82 and 2.72 (3.05 and 3.03 with its larger members by hipMemcpy).
constexpr int kSmallWide = 2048, kSmallNarrow = 4096, kMemberCopy = 16384;
constexpr int kSmallWave = 128; // values per wave
constexpr size_t small_copy_bytes(int values) // pinned memory; values a multiple of kSmallWave
{
   return sizeof(double) * (size_t)values + sizeof(uint32_t) * (size_t)(values / kSmallWave);
}

// The copies of one context: not for two threads at a time, as the context.
struct SmallCopy {
   int wide = kSmallWide, narrow = kSmallNarrow; // largest fields, FP64 and FP32 on the device
   double *buffer = nullptr;
   uint32_t *counts = nullptr;
   uint32_t seq = 0;
   void init(void *pinned); // small_copy_bytes(narrow), aligned to 16
   bool takes(size_t n, bool fp32) const { return n <= (size_t)(fp32 ? narrow : wide); }
   // Complete on return; after the stream's earlier work.
   hipError_t upload(const double *host, void *device, bool fp32, int n, hipStream_t st);
   hipError_t download(void *device, double *host, bool fp32, int n, hipStream_t st);

 private:
   hipError_t wait(int n, hipStream_t st);
};

} // namespace lgpu
