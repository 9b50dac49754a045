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

// Fields of up to this many values are copied by a kernel between pinned memory
// and the device, waited for by its count.  Upload and download, hipMemcpy /
// so: 126 values 11.5 and 11.7 / 7.8 and 7.0 us, 1,000 14.5 and 14.7 / 8.2 and
// 7.6, 2,198 8.9 and 8.5 / 9.0 and 8.5, 9,262 9.9 and 10.8 / 11.6 and 13.4 (it
// takes another path above 16 KiB).
constexpr int kSmallCopy = 2048;
constexpr int kSmallWave = 128;                         // values per wave
constexpr int kSmallWaves = kSmallCopy / kSmallWave;
constexpr size_t kSmallCopyBytes = sizeof(double) * kSmallCopy + sizeof(uint32_t) * kSmallWaves;

// The copies of one context: not for two threads at a time, as the context.
struct SmallCopy {
   double *buffer = nullptr;   // kSmallCopyBytes of pinned memory, counts zero
   uint32_t *counts = nullptr;
   uint32_t seq = 0;
   void init(void *pinned);
   // Complete on return; after the stream's earlier work.  narrow: the device's
   // values are FP32.
   hipError_t upload(const double *host, void *device, bool narrow, int n, hipStream_t st);
   hipError_t download(const void *device, double *host, bool narrow, int n, hipStream_t st);

 private:
   hipError_t wait(int n, hipStream_t st);
};

} // namespace lgpu
