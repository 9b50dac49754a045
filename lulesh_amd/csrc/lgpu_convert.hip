// lgpu_convert.hip -- copies of fields by kernels (lgpu_convert.h).
//
// FP64 <-> FP32: 12 bytes a value and one conversion: bound by memory, so a grid that fills
// the chip with one value a thread and coalesced 8- and 4-byte accesses.
// A field of 7.1 M values, pinned host memory: upload 2.80 ms with the
// conversion on the host, 1.02 ms here (55 GB/s, the link), download 3.71 and
// 1.03 ms.
#include <algorithm>
#include <cstring>

#include "lgpu_convert.h"
#include "lgpu_wait.h"

namespace lgpu {
namespace {

template <typename S, typename D>
__global__ void __launch_bounds__(256) k_convert(const S *__restrict__ src, D *__restrict__ dst, int64_t n)
{
   const int64_t stride = (int64_t)gridDim.x * 256;
   for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) dst[i] = (D)src[i];
}

template <typename S, typename D>
hipError_t launch(const S *src, D *dst, int64_t n, hipStream_t st)
{
   if (n <= 0) return hipSuccess;
   const unsigned grid = (unsigned)std::min<int64_t>((n + 255) / 256, 65536);
   hipLaunchKernelGGL((k_convert<S, D>), dim3(grid), dim3(256), 0, st, src, dst, n);
   return hipGetLastError();
}

// A small field between pinned memory and the device: bound by the latency of
// the link, so one wave a workgroup and two values a lane, 16 bytes of the
// link, all of them in flight at once on many CUs (a workgroup of 1,024
// threads instead: 1,000 values 14.4 us up, 12.3 down).  Each wave stores its
// count when its values are where they belong.
template <bool kUpload, typename T>
__global__ void __launch_bounds__(64) k_small(double2 *__restrict__ pinned, T *__restrict__ device, int n,
                                              uint32_t *counts, uint32_t seq)
{
   const int pair = (int)blockIdx.x * 64 + (int)threadIdx.x, i = 2 * pair;
   if (i < n) {
      const bool two = i + 1 < n;
      if constexpr (kUpload) {
         const double2 v = pinned[pair]; // the buffer holds an even number of values
         device[i] = (T)v.x;
         if (two) device[i + 1] = (T)v.y;
      } else {
         pinned[pair] = double2{(double)device[i], two ? (double)device[i + 1] : 0.0};
      }
   }
   if (threadIdx.x == 0)
      __hip_atomic_store(counts + blockIdx.x, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <bool kUpload, typename T>
hipError_t launch_small(double *pinned, T *device, int n, uint32_t *counts, uint32_t seq, hipStream_t st)
{
   if (n <= 0) return hipSuccess;
   hipLaunchKernelGGL((k_small<kUpload, T>), dim3((unsigned)((n + kSmallWave - 1) / kSmallWave)), dim3(64), 0,
                      st, reinterpret_cast<double2 *>(pinned), device, n, counts, seq);
   return hipGetLastError();
}

} // namespace

void SmallCopy::init(void *pinned)
{
   buffer = static_cast<double *>(pinned);
   counts = reinterpret_cast<uint32_t *>(buffer + limit);
   std::fill(counts, counts + limit / kSmallWave, 0u);
}

hipError_t SmallCopy::wait(int n, hipStream_t st)
{
   for (int w = 0; w * kSmallWave < n; ++w)
      if (!host_reached(counts + w, seq)) return hipStreamSynchronize(st);
   return hipSuccess;
}

hipError_t SmallCopy::upload(const double *host, void *device, bool fp32, int n, hipStream_t st)
{
   std::memcpy(buffer, host, sizeof(double) * (size_t)n);
   ++seq;
   const hipError_t e = fp32 ? launch_small<true>(buffer, static_cast<float *>(device), n, counts, seq, st)
                               : launch_small<true>(buffer, static_cast<double *>(device), n, counts, seq, st);
   return e == hipSuccess ? wait(n, st) : e;
}

hipError_t SmallCopy::download(void *device, double *host, bool fp32, int n, hipStream_t st)
{
   ++seq;
   const hipError_t e = fp32 ? launch_small<false>(buffer, static_cast<float *>(device), n, counts, seq, st)
                               : launch_small<false>(buffer, static_cast<double *>(device), n, counts, seq, st);
   if (e != hipSuccess) return e;
   const hipError_t w = wait(n, st);
   if (w == hipSuccess) std::memcpy(host, buffer, sizeof(double) * (size_t)n);
   return w;
}

bool converts_on_device(const void *host, int64_t n, bool upload)
{
   constexpr int64_t kPinnedUp = 150000, kPinnedDown = 98304, kUp = 1 << 20; // converted on the host
   if (n <= (upload ? kPinnedUp : kPinnedDown)) return false;
   hipPointerAttribute_t a{};
   if (hipPointerGetAttributes(&a, host) != hipSuccess) {
      (void)hipGetLastError(); // memory that the runtime does not know
      a.type = hipMemoryTypeUnregistered;
   }
   return a.type == hipMemoryTypeHost || (upload && n > kUp);
}

hipError_t launch_narrow(const double *src, float *dst, int64_t n, hipStream_t st)
{
   return launch(src, dst, n, st);
}

hipError_t launch_widen(const float *src, double *dst, int64_t n, hipStream_t st)
{
   return launch(src, dst, n, st);
}

} // namespace lgpu
