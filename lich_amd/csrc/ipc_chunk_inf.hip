// ipc_chunk_inf.hip - k-chunk kernel, inference update (layout INF).
#include "ipc_chunk_kernel.h"

namespace ipc {

hipError_t launch_chunk_inf(const GemmProblem* probs, int count, int storage, int operand, int tile, hipStream_t s) {
  if (storage == DT_F32) {
    if (operand == DT_F32) return chunk::run_chunks<float, float, LAYOUT_INF, 1>(probs, count, tile, s);
    if (operand == DT_F16) return chunk::run_chunks<float, f16, LAYOUT_INF, 1>(probs, count, tile, s);
    return chunk::run_chunks<float, bf16, LAYOUT_INF, 1>(probs, count, tile, s);
  }
  if (storage == DT_F16) return chunk::run_chunks<f16, f16, LAYOUT_INF, 1>(probs, count, tile, s);
  return chunk::run_chunks<bf16, bf16, LAYOUT_INF, 1>(probs, count, tile, s);
}

}  // namespace ipc
