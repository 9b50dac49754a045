// lgpu_convert.h -- conversion between the FP64 fields of the ABI and the
// fields the mixed form stores in FP32 (p, q, ss and the Q gradients), on the
// device.
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

} // namespace lgpu
