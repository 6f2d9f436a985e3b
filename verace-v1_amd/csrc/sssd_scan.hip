// Kernel-family selection for the prefill scan:
//   bf16/fp16 I/O, head_dim 128, T >= 32  -> chunk-parallel MFMA scan (sssd_chunk.hip)
//   T == 1, head_dim 128 (any I/O dtype)   -> persistent single-step kernel (sssd_step.hip)
//   head_dim <= 128, T >= chunk32_min_tokens (5 .. 20 by heads, head_dim and type)
//                                          -> chunked fp32 MFMA scan (sssd_chunk32.hip), given its
//                                             workspace
//   everything else (head_dim > 128, fewer tokens, no workspace) -> token-sequential fp32 scan
//                                             (sssd_seq.hip)
#include "vmi_common.h"
#include "vmi_dispatch.h"

namespace vmi {

size_t scan_workspace_required(int64_t B, int64_t T, int64_t H, int64_t D, int io_dtype) {
  return chunk_workspace_bytes(B, T, H, D, io_dtype);
}

size_t scan_workspace_bytes(int64_t B, int64_t T, int64_t H, int64_t D, int io_dtype) {
  if (use_chunk_path(T, D, io_dtype)) return chunk_workspace_bytes(B, T, H, D, io_dtype);
  return chunk32_workspace_bytes(B, T, H, D, io_dtype);
}

hipError_t dispatch_scan(const void* q, const void* k, const void* v, const void* delta,
                         int io_dtype, int delta_dtype, const float* psi_in, void* out,
                         float* psi_out, int B, int T, int H, int D, void* workspace,
                         size_t workspace_bytes, hipStream_t stream) {
  if (use_chunk_path(T, D, io_dtype))
    return launch_sssd_chunked(q, k, v, delta, io_dtype, delta_dtype, psi_in, out, psi_out, B, T,
                               H, workspace, stream);
  if (use_step128(T, D))
    return launch_sssd_step128(q, k, v, delta, io_dtype, delta_dtype, psi_in, out, psi_out,
                               B, H, stream);
  if (use_chunk32(static_cast<int64_t>(B) * H, T, D, io_dtype) && workspace != nullptr &&
      workspace_bytes >= chunk32_workspace_bytes(B, T, H, D, io_dtype) &&
      reinterpret_cast<uintptr_t>(workspace) % 16 == 0)
    return launch_sssd_chunk32(q, k, v, delta, io_dtype, delta_dtype, psi_in, out, psi_out, B, T, H,
                               D, workspace, stream);
  return launch_sssd_seq(q, k, v, delta, io_dtype, delta_dtype, psi_in, out, psi_out, B, T, H, D,
                         stream);
}

}  // namespace vmi
