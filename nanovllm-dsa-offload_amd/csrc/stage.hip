// Staging of a decode step's inputs into the fixed-address buffers of a
// captured graph: up to kMaxStageItems row-wise copies with padding in one
// launch.
//
// Each item copies `src_bytes` of every real row and fills the rest of the
// row, and the rows after the real ones, with a 32-bit pattern.  The copies
// are tiny (a batch of one: 12 buffers, most of them 4 bytes), so their cost
// is the launches: about twenty copies and fills per step, against a captured
// layer-step of 47 us.  One launch (4.5 us) moves all of them, in units of 16
// bytes where addresses and widths allow it: a replay with new inputs for one
// request of 20480 tokens takes 56 us instead of 112 to 131 (host-bound, by
// the host).
#include "nvdsa_common.h"
#include "nvdsa_kernels.h"

namespace nvdsa {
namespace {

constexpr int kStageThreads = 256;
constexpr int kStageUnits = 4;  // units per thread

template <typename U>
__device__ __forceinline__ void stage_units(const StageItem& it, int64_t first, U fill) {
  const int64_t row_units = it.dst_bytes / sizeof(U), src_units = it.src_bytes / sizeof(U);
  const int64_t total = it.rows * row_units;
#pragma unroll
  for (int k = 0; k < kStageUnits; ++k) {
    const int64_t i = first + k * kStageThreads;
    if (i >= total) return;
    const int64_t row = i / row_units, col = i - row * row_units;
    U v = fill;
    if (row < it.real && col < src_units)
      v = reinterpret_cast<const U*>(static_cast<const char*>(it.src) + row * it.src_stride)[col];
    static_cast<U*>(it.dst)[i] = v;
  }
}

__global__ __launch_bounds__(kStageThreads) void stage_inputs_kernel(StageArgs a) {
  int item = 0;
  while (item + 1 < a.count && static_cast<int>(blockIdx.x) >= a.first_block[item + 1]) ++item;  // (uniform)
  const StageItem& it = a.items[item];
  const int64_t first = static_cast<int64_t>(blockIdx.x - a.first_block[item]) * kStageThreads * kStageUnits + threadIdx.x;
  const uint32_t f = static_cast<uint32_t>(it.fill);
  if (it.unit == 16)
    stage_units(it, first, u32x4_t{f, f, f, f});
  else if (it.unit == 4)
    stage_units(it, first, f);
  else
    stage_units(it, first, static_cast<uint16_t>(f));
}

}  // namespace

hipError_t launch_stage_inputs(StageArgs& a, hipStream_t stream) {
  int64_t blocks = 0;
  for (int i = 0; i < a.count; ++i) {
    StageItem& it = a.items[i];
    const uintptr_t all = reinterpret_cast<uintptr_t>(it.dst) | reinterpret_cast<uintptr_t>(it.src) |
                          static_cast<uintptr_t>(it.dst_bytes) | static_cast<uintptr_t>(it.src_bytes) |
                          static_cast<uintptr_t>(it.src_stride);
    it.unit = (all & 15) == 0 ? 16 : (all & 3) == 0 ? 4 : 2;
    a.first_block[i] = static_cast<int32_t>(blocks);
    blocks += ceil_div(it.rows * it.dst_bytes / it.unit, kStageThreads * kStageUnits);
    if (blocks >= (int64_t{1} << 23)) return hipErrorInvalidValue;
  }
  if (blocks == 0) return hipSuccess;
  launch_kernel(kKernStage, stage_inputs_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kStageThreads), stream, a);
  return hipGetLastError();
}

}  // namespace nvdsa
