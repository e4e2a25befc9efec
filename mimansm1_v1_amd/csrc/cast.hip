// fp32 -> bf16 (round to nearest even) of up to four tensors into one buffer,
// one after the other, in one launch: the operand casts of a projection
// (activations and the weights wq | wk | wv), which torch runs as one launch
// each plus a concatenation (CODE/mimans/model/attention_tilelang.py:470-487
// under autocast).  HBM-bound; 8 values per thread and step.
#include <hip/hip_runtime.h>

#include "mm1_common.h"

namespace mm1 {

struct CastSegments {
  const float* src[4];
  long end8[4];       // first 8-value group past each segment
};

__global__ __launch_bounds__(256) void cast_bf16_kernel(const CastSegments s, __bf16* __restrict__ dst) {
  const long total = s.end8[3], stride = (long)gridDim.x * 256;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < total; i += stride) {
    const int seg = (i >= s.end8[0]) + (i >= s.end8[1]) + (i >= s.end8[2]);
    const float* p = s.src[0];
    long first = 0;
#pragma unroll
    for (int j = 1; j < 4; ++j) {
      if (seg == j) {
        p = s.src[j];
        first = s.end8[j - 1];
      }
    }
    const f32x4 a = *reinterpret_cast<const f32x4*>(p + 8 * (i - first));
    const f32x4 b = *reinterpret_cast<const f32x4*>(p + 8 * (i - first) + 4);
    bf16x8 r;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      r[t] = (__bf16)a[t];
      r[4 + t] = (__bf16)b[t];
    }
    *reinterpret_cast<bf16x8*>(dst + 8 * i) = r;
  }
}

hipError_t launch_cast_bf16(const float* const src[4], const long n[4], void* dst, hipStream_t stream) {
  CastSegments s;
  long end = 0;
  for (int j = 0; j < 4; ++j) {
    s.src[j] = src[j];
    end += n[j] / 8;
    s.end8[j] = end;
  }
  const long blocks = (end + 255) / 256;
  hipLaunchKernelGGL(cast_bf16_kernel, dim3((unsigned)(blocks < 16384 ? blocks : 16384)), dim3(256), 0, stream, s,
                     static_cast<__bf16*>(dst));
  return hipGetLastError();
}

}  // namespace mm1
