// ipc_chunk_wgt.hip - k-chunk kernel, weight update (layout WGT).
#include "ipc_chunk_kernel.h"

namespace ipc {

hipError_t launch_chunk_wgt(const GemmProblem* probs, int count, int storage, int operand, int tile, hipStream_t s) {
  if (storage == DT_F32) {
    if (operand == DT_F32) return chunk::run_chunks<float, float, LAYOUT_WGT, 1>(probs, count, tile, s);
    if (operand == DT_F16) return chunk::run_chunks<float, f16, LAYOUT_WGT, 1>(probs, count, tile, s);
    return chunk::run_chunks<float, bf16, LAYOUT_WGT, 1>(probs, count, tile, s);
  }
  if (storage == DT_F16) return chunk::run_chunks<f16, f16, LAYOUT_WGT, 1>(probs, count, tile, s);
  return chunk::run_chunks<bf16, bf16, LAYOUT_WGT, 1>(probs, count, tile, s);
}

}  // namespace ipc
