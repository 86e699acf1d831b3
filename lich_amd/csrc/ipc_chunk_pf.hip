// ipc_chunk_pf.hip - k-chunk kernel, prediction + error and forward (layout PF).
#include "ipc_chunk_kernel.h"

namespace ipc {

template <typename OT>
static hipError_t pf_split(const GemmProblem* probs, int count, int split, int tile, hipStream_t s) {
  switch (split) {
    case 2: return chunk::run_chunks<float, OT, LAYOUT_PF, 2>(probs, count, tile, s);
    case 3: return chunk::run_chunks<float, OT, LAYOUT_PF, 3>(probs, count, tile, s);
    default: return chunk::run_chunks<float, OT, LAYOUT_PF, 1>(probs, count, tile, s);
  }
}

hipError_t launch_chunk_pf(const GemmProblem* probs, int count, int storage, int operand, int split, int tile,
                           hipStream_t s) {
  if (storage == DT_F32) {
    if (operand == DT_F32) return chunk::run_chunks<float, float, LAYOUT_PF, 1>(probs, count, tile, s);
    if (operand == DT_F16) return pf_split<f16>(probs, count, split, tile, s);
    return pf_split<bf16>(probs, count, split, tile, s);
  }
  if (storage == DT_F16) return chunk::run_chunks<f16, f16, LAYOUT_PF, 1>(probs, count, tile, s);
  return chunk::run_chunks<bf16, bf16, LAYOUT_PF, 1>(probs, count, tile, s);
}

}  // namespace ipc
