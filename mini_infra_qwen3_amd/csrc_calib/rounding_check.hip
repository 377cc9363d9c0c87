// Check of the kernels' bf16 rounding (mi_common.h) against the integer construction it stands for, built with
// the kernels' flags.  Not part of the paged-KV C ABI: it lives in libmi_calib.so, for the tests.
#include "../csrc/mi_common.h"

namespace {

// Round to nearest even on the bits: add 0x7fff plus the lowest kept bit, truncate; a NaN keeps its payload's high
// half with the quiet bit set.
__device__ uint32_t integer_bf16(uint32_t u) {
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// Counts the fp32 patterns [first, first + count) at which a helper differs from the construction.
__global__ void round_patterns(uint64_t first, uint64_t count, unsigned long long* bad) {
  const uint64_t step = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  unsigned long long mine = 0;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += step) {
    const uint32_t u = static_cast<uint32_t>(first + i);
    const float f = __uint_as_float(u);
    const uint32_t want = integer_bf16(u);
    const uint32_t pair = mi::pack_bf16x2(f, f);
    mine += (mi::f32_to_bf16_bits(f) & 0xffffu) != want || pair != (want | (want << 16)) ||
            __float_as_uint(mi::round_bf16(f)) != want << 16;
  }
  if (mine) atomicAdd(bad, mine);
}

// Double -> float -> bf16, as the exact kernels' chains round: in[i] through the helpers against the same two
// roundings with the float made opaque between them, so that nothing can fold them into one.
__global__ void round_doubles(const double* in, uint64_t count, unsigned long long* bad) {
  const uint64_t step = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  unsigned long long mine = 0;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += step) {
    const double d = in[i];
    const uint32_t bits = mi::f32_to_bf16_bits(static_cast<float>(d)) & 0xffffu;
    const uint32_t scaled = __float_as_uint(mi::round_bf16(mi::round_bf16(static_cast<float>(d)) * 0.5f));
    float f = static_cast<float>(d);
    asm volatile("" : "+v"(f));
    const uint32_t want = integer_bf16(__float_as_uint(f));
    float g = __uint_as_float(want << 16) * 0.5f;
    asm volatile("" : "+v"(g));
    mine += bits != want || scaled != integer_bf16(__float_as_uint(g)) << 16;
  }
  if (mine) atomicAdd(bad, mine);
}

}  // namespace

// bad: one device counter, zeroed by the caller.  Returns the HIP error of the launch.
extern "C" int32_t calib_round_patterns(uint64_t first, uint64_t count, void* bad, void* stream) {
  if (count == 0 || count > (1ull << 32) - first || bad == nullptr) return -1;
  round_patterns<<<4096, 256, 0, mi::as_stream(stream)>>>(first, count, static_cast<unsigned long long*>(bad));
  return hipGetLastError();
}
extern "C" int32_t calib_round_doubles(const void* in, uint64_t count, void* bad, void* stream) {
  if (count == 0 || in == nullptr || bad == nullptr) return -1;
  round_doubles<<<1024, 256, 0, mi::as_stream(stream)>>>(static_cast<const double*>(in), count,
                                                         static_cast<unsigned long long*>(bad));
  return hipGetLastError();
}
