// gemm_core.hpp -- what the 256x256 GEMM kernels (dense bf16, fp8, general)
// share besides the pipelined tile itself (gemm_pipe.hpp): the tile order
// and launch plan (tile_plan.hpp), the choice of epilogue and the empty sum.
#pragma once

#include "common.hpp"
#include "tile_plan.hpp"

namespace gemm_core {

// The workgroup-to-tile order and the tail-quarter mapping (tile_plan.hpp).
using tile_plan::tail_quarter;
using tile_plan::xcd_tile_order;

// Host: whether a 256x256-tile launch whose operands (A and B together) take
// `operand_bytes` stores C through LDS (gemm_pipe::store_bf16_staged).  C
// written straight from the accumulators lands in the caches in part-lines;
// once the operands alone nearly fill the 256 MiB last-level cache, that C
// evicts operand panels that later tiles re-read, and the staged nontemporal
// store is faster (measured: +9% bf16 8192^3, +15% 1024x28672x4096).  With
// smaller operands the staging only adds ~1 us per tile (-1% to -8% on eight
// shapes from 4096^3 to 8192x8192x1024, bf16 and fp8).
constexpr uint64_t kStagedOperandBytes = 192ull << 20;
inline bool staged_epilogue(uint64_t operand_bytes) {
  return operand_bytes >= kStagedOperandBytes;
}

// K = 0: C is all +0 (an empty sum), whatever else the call scales it by.  A
// grid-stride fill kernel rather than a memset node, so a caller may capture
// the launch in a HIP graph.
namespace {
template <class T>
__global__ void __launch_bounds__(256) zero_fill_kernel(T* __restrict__ c, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) c[i] = 0;
}
}  // namespace
inline dim3 zero_fill_grid(uint64_t n) {
  const uint64_t blocks = (n + 255u) / 256u;
  return dim3((unsigned)(blocks < 4096u ? blocks : 4096u));
}

}  // namespace gemm_core
