// Rounding of float32 op inputs to fp16.
//
// The ops take float32 tensors (the reference's CPU paths compute in fp32,
// MInference-NPU/minference/ops/streaming_kernel_npu.py:138-144) and run on
// their roundings: fp16 when every finite value fits its range, else bf16.
// One pass reads each tensor once, writes its fp16 rounding (nearest even)
// and raises *flag when a finite value lies beyond fp16's range.  The flag is
// written in that case only, so it can live in host memory: no reduction, no
// copy back.
//
// Bound by memory: 4 bytes read and 2 written per element; thread = 8
// elements (two 16-byte loads, one 16-byte store).  Three tensors of 32 x
// 4096 x 96 (226 MB in all) in one launch; the library ops it replaces (abs,
// isfinite, where, amax, the conversion and a host read, each per tensor) took
// 31 launches and three waits: streaming_forward on them 483 us, now 122 us.

#include "msa_kernels.h"

namespace msa {

namespace {

typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2v __attribute__((ext_vector_type(2)));

__global__ __launch_bounds__(256) void round_f16_kernel(const RoundParams P) {
  const RoundTensor& t = P.t[blockIdx.y];
  const uint32_t u = blockIdx.x * 256u + threadIdx.x;  // 8-element unit of the tensor
  if (u >= t.units) return;
  const uint32_t row = u / t.upr, c = u - row * t.upr;  // units per row
  const uint32_t bh = row / t.s, s = row - bh * t.s;
  const uint32_t b = bh / t.h, h = bh - b * t.h;
  const float* src = t.src + b * t.sb + h * t.sh + s * t.ss + 8 * c;
  const float4 x = *reinterpret_cast<const float4*>(src);
  const float4 y = *reinterpret_cast<const float4*>(src + 4);
  const float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
  u32x4 o;
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    m = fmaxf(m, fmaxf(finite_abs(v[2 * i]), finite_abs(v[2 * i + 1])));
    o[i] = __builtin_bit_cast(uint32_t,
                              __builtin_convertvector(f32x2v{v[2 * i], v[2 * i + 1]}, f16x2v));
  }
  store16(t.dst + uint64_t(u) * 8, o);
  if (m > kF16Max) __hip_atomic_store(P.flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

hipError_t launch_round(const RoundParams& p, int n, hipStream_t st) {
  uint32_t most = 0;
  for (int i = 0; i < n; ++i) most = p.t[i].units > most ? p.t[i].units : most;
  hipLaunchKernelGGL(round_f16_kernel, dim3(most / 256 + (most % 256 != 0), n), dim3(256), 0, st, p);
  return hipGetLastError();
}

}  // namespace msa
