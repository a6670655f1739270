// Non-finite scan of up to three tensors in one launch: the check of the
// reference's host fix-up (adasplashattention.cu:599-606, :684-697), which
// reads one word back instead of two reductions per tensor (isnan, any,
// copy, isinf, any, copy).  HBM-bound: each tensor is read once, 16 bytes
// per lane.  Measured with the read-back at 1x6x1500x64 fp32, three
// gradients: 204 -> 26 us; one tensor 64 -> 26 us.
#include <type_traits>

#include "asa_device.hpp"
#include "asa_launch.hpp"

namespace asa {
namespace {

constexpr int kThreads = 256;

// Bits of `w` (one fp32 or two 16-bit values): 1 a NaN, 2 an infinity.
template <typename T>
__device__ __forceinline__ uint32_t word_flags(uint32_t w) {
  if constexpr (std::is_same<T, float>::value) {
    const uint32_t a = w & 0x7fffffffu;
    return (a > 0x7f800000u ? 1u : 0u) | (a == 0x7f800000u ? 2u : 0u);
  } else {
    constexpr uint32_t kInf = std::is_same<T, u16>::value ? 0x7f80u : 0x7c00u;
    const uint32_t a = w & 0x7fffu, b = (w >> 16) & 0x7fffu;
    return (a > kInf || b > kInf ? 1u : 0u) | (a == kInf || b == kInf ? 2u : 0u);
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void nonfinite_kernel(NonfiniteParams p) {
  const int i = blockIdx.y;
  constexpr int kEpc = 16 / int(sizeof(T));
  const size_t n = p.n[i], chunks = n / kEpc;
  const uint4* src = static_cast<const uint4*>(p.t[i]);
  uint32_t f = 0;
  for (size_t c = size_t(blockIdx.x) * kThreads + threadIdx.x; c < chunks; c += size_t(gridDim.x) * kThreads) {
    const uint4 v = src[c];
    f |= word_flags<T>(v.x) | word_flags<T>(v.y) | word_flags<T>(v.z) | word_flags<T>(v.w);
  }
  if (blockIdx.x == 0 && threadIdx.x < n - chunks * kEpc) {  // the tail's elements
    const T* e = static_cast<const T*>(p.t[i]) + chunks * kEpc + threadIdx.x;
    if constexpr (sizeof(T) == 4) f |= word_flags<T>(*reinterpret_cast<const uint32_t*>(e));
    else f |= word_flags<T>(*reinterpret_cast<const uint16_t*>(e));
  }
  if (f) atomicOr(p.flags, f << (2 * i));
}

}  // namespace

hipError_t launch_nonfinite(const NonfiniteParams& p, int dtype, hipStream_t s) {
  size_t most = 0;
  for (int i = 0; i < p.count; ++i) most = p.n[i] > most ? p.n[i] : most;
  const size_t per = size_t(kThreads) * 16 / elem_bytes(dtype);
  const size_t want = (most + per - 1) / per;
  const dim3 grid(unsigned(want < 1 ? 1 : want > 2048 ? 2048 : want), unsigned(p.count));
  if (dtype == kElemBF16) hipLaunchKernelGGL(nonfinite_kernel<u16>, grid, dim3(kThreads), 0, s, p);
  else if (dtype == kElemF16) hipLaunchKernelGGL(nonfinite_kernel<h16>, grid, dim3(kThreads), 0, s, p);
  else hipLaunchKernelGGL(nonfinite_kernel<float>, grid, dim3(kThreads), 0, s, p);
  return hipGetLastError();
}

}  // namespace asa
