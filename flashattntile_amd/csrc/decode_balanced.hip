// decode_balanced.hip -- the balanced instantiations of the decode kernels
// (decode_kernels.h): equal runs of the batch's work per 4-wave workgroup.
#include "decode_kernels.h"

namespace {

template <typename QT, int KV, int D, bool LANE>
void launch_valu_t(const fat::DecodeParams& prm, dim3 grid, hipStream_t stream) {
  hipLaunchKernelGGL((fat::paged_decode_kernel<QT, KV, D, 4, 4, LANE, true>), grid, dim3(256), 0, stream, prm);
}

template <typename QT, int KV>
void launch_lane_kv(const fat::DecodeParams& prm, int D, dim3 grid, hipStream_t stream) {
  if constexpr (KV == fat::KV_SAME) {
    if (D == 32) return launch_valu_t<QT, KV, 32, true>(prm, grid, stream);
  } else {
    if (D == 256) return launch_valu_t<QT, KV, 256, true>(prm, grid, stream);
  }
  if (D == 128) launch_valu_t<QT, KV, 128, true>(prm, grid, stream);
  else launch_valu_t<QT, KV, 64, true>(prm, grid, stream);
}

template <typename QT, int KV>
void launch_kv(const fat::DecodeParams& prm, bool lane, int D, dim3 grid, hipStream_t stream) {
  if (lane) return launch_lane_kv<QT, KV>(prm, D, grid, stream);
  if constexpr (KV == fat::KV_SAME) {
    if (D == 128) launch_valu_t<QT, KV, 128, false>(prm, grid, stream);
    else launch_valu_t<QT, KV, 64, false>(prm, grid, stream);
  } else if (D == 128) {
    hipLaunchKernelGGL((fat::paged_decode_mfma_kernel<QT, KV, 128, 4, true>), grid, dim3(256), 0, stream, prm);
  } else {
    hipLaunchKernelGGL((fat::paged_decode_mfma_kernel<QT, KV, 64, 4, true>), grid, dim3(256), 0, stream, prm);
  }
}

template <typename QT>
void launch_q(const fat::DecodeParams& prm, int kv, bool lane, int D, dim3 grid, hipStream_t stream) {
  switch (kv) {
    case fat::KV_SAME: launch_kv<QT, fat::KV_SAME>(prm, lane, D, grid, stream); break;
    case fat::KV_I8: launch_kv<QT, fat::KV_I8>(prm, lane, D, grid, stream); break;
    default: launch_kv<QT, fat::KV_FP8>(prm, lane, D, grid, stream); break;
  }
}

}  // namespace

namespace fat_host {

int launch_decode_balanced(const fat::DecodeParams& prm, int q_dtype, int kv, bool lane, int head_dim, int groups,
                           hipStream_t stream) {
  const dim3 grid((unsigned)groups);
  if (q_dtype == FAT_DTYPE_F16) launch_q<fat::F16>(prm, kv, lane, head_dim, grid, stream);
  else if (q_dtype == FAT_DTYPE_BF16) launch_q<fat::BF16>(prm, kv, lane, head_dim, grid, stream);
  else launch_lane_kv<fat::F32, fat::KV_SAME>(prm, head_dim, grid, stream);
  return launch_status("balanced decode kernel");
}

}  // namespace fat_host
