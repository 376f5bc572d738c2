// decode.hip -- single-query paged decode for gfx950 (fp16/bf16/int8/fp8 K/V).
//
// Behaviour follows the FlashAttnTile decode path:
//   flashattn_tile/kernels/decode.py:47-127   (_decode_paged_kernel)
//   flashattn_tile/kernels/decode.py:223-356  (split kernel + LSE reduce)
//   flashattn_tile/kernels/decode.py:359-447  (quantised K/V)
// Design (MI355X-first, not a translation of the Triton programs):
//   * one workgroup per (split, GQA head group, sequence); the HG query heads
//     of a group share one KV head, so every K/V page is read from HBM once
//     per group instead of once per query head;
//   * a wave streams 16-token units (32 at fp16/bf16 head_dim 64); lane
//     (r, c) owns row r of each 16-byte wide load and dims
//     [c*EPL, c*EPL+EPL); K and V rows arrive as global_load_dwordx4, one
//     unit ahead of the compute (register double buffer);
//   * q.k partial sums are reduced across the LPR lanes of a row with a
//     transposing DPP butterfly that leaves one (head, token) score per lane;
//   * softmax state (running max m, sum l) is shared by the whole wave; the
//     probabilities are broadcast to the PV lanes through a few bytes of LDS;
//   * PV accumulates in fp32 (no rounding of p), matching the fp32 oracle;
//   * int8/fp8 pages are dequantised in registers as
//     round_to_q_dtype(float(x) * scale), the reference's own
//     dequantise-then-attend semantics (flashattn_tile/quant.py:145-161);
//     with fp16 queries K is staged exact and k_scale multiplies the fp32
//     scores (the reference's quantised kernel, kernels/decode.py:419-429),
//     and the MFMA decode forms int8 V as x * fp16(scale) (k8_exact_f16);
//   * with split_k > 1 each workgroup writes (acc, m, l) for its partition
//     and a second kernel merges the partitions by log-sum-exp;
//   * multi-token decode (q_len = T > 1, e.g. speculative verification) runs
//     on the MFMA kernel: its 32 MFMA columns are (query head, token) rows,
//     G * T of them per KV head, so each K/V page is still read once per KV
//     head per 32 rows; token t sees keys j <= seq_len - T + t (the
//     bottom-right causal convention of flashattn_tile/reference.py:19-22).
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "decode_kernels.h"

namespace fat {

// Log-sum-exp merge of split-K partitions (decode.py:316-356 semantics):
//   M = max_s m_s, w_s = 2^(m_s - M), o = sum_s acc_s w_s / sum_s l_s w_s.
// Rows are (sequence, token, head) with T tokens per sequence: one launch
// per decode (decode_merge_kernel), or inside the decode launch by its last
// partition (merge_in_launch), with the same arithmetic.
template <typename QT, int SMAX>
__global__ __launch_bounds__(256) void decode_merge_kernel(const float* __restrict__ ws_acc,
                                                           const float* __restrict__ ws_ml, uint8_t* out,
                                                           int B, int T, int H, int D, int S, int64_t o_sb,
                                                           int64_t o_st, int64_t o_sh) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)B * T * H * D) return;
  const int d = idx % D;
  const int64_t bh = idx / D;
  const int h = bh % H;
  const int64_t bt = bh / H;
  const int t = bt % T;
  const int b = bt / T;
  merge_elem<QT, SMAX>(ws_acc, ws_ml, bh, d, D, S, out, (int64_t)b * o_sb + (int64_t)t * o_st + (int64_t)h * o_sh + d);
}

}  // namespace fat

// ===========================================================================
// Host side
// ===========================================================================
namespace {

int ilog2_exact(int x) {
  if (x <= 0 || (x & (x - 1))) return -1;
  int l = 0;
  while ((1 << l) < x) ++l;
  return l;
}

template <typename QT, int KV, int D, int HG>
int launch_decode_t(const fat::DecodeParams& prm, int nw, dim3 grid, hipStream_t stream) {
  if (nw == 8) {
    hipLaunchKernelGGL((fat::paged_decode_kernel<QT, KV, D, HG, 8>), grid, dim3(8 * 64), 0, stream, prm);
  } else {
    hipLaunchKernelGGL((fat::paged_decode_kernel<QT, KV, D, HG, 4>), grid, dim3(4 * 64), 0, stream, prm);
  }
  return fat_host::launch_status("paged_decode_kernel");
}

// 8-bit caches take the VALU kernel only with 4-head groups: the 8-head
// instantiations with in-register dequantisation spill (the MFMA kernel is
// the library's choice for 8-bit caches anyway).
template <typename QT, int KV>
int launch_decode_kv(const fat::DecodeParams& prm, int D, int HG, int nw, dim3 grid, hipStream_t stream) {
  if constexpr (KV == fat::KV_SAME) {
    if (HG == 8)
      return D == 128 ? launch_decode_t<QT, KV, 128, 8>(prm, nw, grid, stream)
                      : launch_decode_t<QT, KV, 64, 8>(prm, nw, grid, stream);
  }
  return D == 128 ? launch_decode_t<QT, KV, 128, 4>(prm, nw, grid, stream)
                  : launch_decode_t<QT, KV, 64, 4>(prm, nw, grid, stream);
}

template <typename QT>
int launch_decode_q(const fat::DecodeParams& prm, int kv, int D, int HG, int nw, dim3 grid,
                    hipStream_t stream) {
  switch (kv) {
    case fat::KV_SAME: return launch_decode_kv<QT, fat::KV_SAME>(prm, D, HG, nw, grid, stream);
    case fat::KV_I8: return launch_decode_kv<QT, fat::KV_I8>(prm, D, HG, nw, grid, stream);
    default: return launch_decode_kv<QT, fat::KV_FP8>(prm, D, HG, nw, grid, stream);
  }
}


// Per-lane addressing (paged_decode_kernel<..., LANE>), 4-head groups.
template <typename QT, int KV, int D>
int launch_lane_t(const fat::DecodeParams& prm, int nw, dim3 grid, hipStream_t stream) {
  if (nw == 8) {
    hipLaunchKernelGGL((fat::paged_decode_kernel<QT, KV, D, 4, 8, true>), grid, dim3(8 * 64), 0, stream, prm);
  } else {
    hipLaunchKernelGGL((fat::paged_decode_kernel<QT, KV, D, 4, 4, true>), grid, dim3(4 * 64), 0, stream, prm);
  }
  return fat_host::launch_status("paged_decode_kernel");
}

// The shapes it is built for: at least four lanes per row (fp16/bf16 and fp32
// from head_dim 32, 8-bit from 64) and a unit's registers without spills
// (head_dim up to 256, fp32 up to 128).
bool lane_takes(int q_dtype, int kv, int D) {
  const int lo = kv == fat::KV_SAME ? 32 : 64;
  return D >= lo && D <= (q_dtype == FAT_DTYPE_F32 ? 128 : 256);
}

template <typename QT, int KV>
int launch_lane_kv(const fat::DecodeParams& prm, int D, int nw, dim3 grid, hipStream_t stream) {
  if constexpr (KV == fat::KV_SAME) {
    if (D == 32) return launch_lane_t<QT, KV, 32>(prm, nw, grid, stream);
  }
  if constexpr (!std::is_same<QT, fat::F32>::value) {
    if (D == 256) return launch_lane_t<QT, KV, 256>(prm, nw, grid, stream);
  }
  return D == 128 ? launch_lane_t<QT, KV, 128>(prm, nw, grid, stream)
                  : launch_lane_t<QT, KV, 64>(prm, nw, grid, stream);
}

template <typename QT>
int launch_lane_q(const fat::DecodeParams& prm, int kv, int D, int nw, dim3 grid, hipStream_t stream) {
  switch (kv) {
    case fat::KV_SAME: return launch_lane_kv<QT, fat::KV_SAME>(prm, D, nw, grid, stream);
    case fat::KV_I8: return launch_lane_kv<QT, fat::KV_I8>(prm, D, nw, grid, stream);
    default: return launch_lane_kv<QT, fat::KV_FP8>(prm, D, nw, grid, stream);
  }
}

int launch_lane(const fat::DecodeParams& prm, int q_dtype, int kv, int D, int nw, dim3 grid, hipStream_t stream) {
  if (q_dtype == FAT_DTYPE_F16) return launch_lane_q<fat::F16>(prm, kv, D, nw, grid, stream);
  if (q_dtype == FAT_DTYPE_BF16) return launch_lane_q<fat::BF16>(prm, kv, D, nw, grid, stream);
  return launch_lane_kv<fat::F32, fat::KV_SAME>(prm, D, nw, grid, stream);
}

template <typename QT, int KV, int NW>
void launch_decode_mfma_kvw(const fat::DecodeParams& prm, int D, dim3 grid, hipStream_t stream) {
  if (D == 128)
    hipLaunchKernelGGL((fat::paged_decode_mfma_kernel<QT, KV, 128, NW>), grid, dim3(NW * 64), 0, stream, prm);
  else
    hipLaunchKernelGGL((fat::paged_decode_mfma_kernel<QT, KV, 64, NW>), grid, dim3(NW * 64), 0, stream, prm);
}

template <typename QT, int KV>
void launch_decode_mfma_kv(const fat::DecodeParams& prm, int D, int nw, dim3 grid, hipStream_t stream) {
  if (nw == 8) launch_decode_mfma_kvw<QT, KV, 8>(prm, D, grid, stream);
  else launch_decode_mfma_kvw<QT, KV, 4>(prm, D, grid, stream);
}

template <typename QT>
void launch_decode_mfma_q(const fat::DecodeParams& prm, int kv, int D, int nw, dim3 grid, hipStream_t stream) {
  switch (kv) {
    case fat::KV_SAME: launch_decode_mfma_kv<QT, fat::KV_SAME>(prm, D, nw, grid, stream); break;
    case fat::KV_I8: launch_decode_mfma_kv<QT, fat::KV_I8>(prm, D, nw, grid, stream); break;
    default: launch_decode_mfma_kv<QT, fat::KV_FP8>(prm, D, nw, grid, stream); break;
  }
}

template <typename QT, int SMAX>
void launch_merge_s(const fat::DecodeParams& prm, const fat_decode_args* a, int D, dim3 mgrid, hipStream_t stream) {
  hipLaunchKernelGGL((fat::decode_merge_kernel<QT, SMAX>), mgrid, dim3(256), 0, stream, prm.ws_acc, prm.ws_ml,
                     prm.out, a->batch, prm.T, a->num_heads, D, a->split_k, a->out_stride_b, prm.o_st,
                     a->out_stride_h);
}

template <typename QT>
void launch_merge_q(const fat::DecodeParams& prm, const fat_decode_args* a, int D, dim3 mgrid, hipStream_t stream) {
  const int S = a->split_k;
  if (S <= 4) launch_merge_s<QT, 4>(prm, a, D, mgrid, stream);
  else if (S <= 8) launch_merge_s<QT, 8>(prm, a, D, mgrid, stream);
  else if (S <= 16) launch_merge_s<QT, 16>(prm, a, D, mgrid, stream);
  else if (S <= 32) launch_merge_s<QT, 32>(prm, a, D, mgrid, stream);
  else launch_merge_s<QT, 64>(prm, a, D, mgrid, stream);  // split_k <= 64 (validated)
}

int launch_merge(const fat::DecodeParams& prm, const fat_decode_args* a, int D, hipStream_t stream) {
  const int64_t n = (int64_t)a->batch * prm.T * a->num_heads * D;
  const dim3 mgrid((unsigned)((n + 255) / 256));
  if (a->q_dtype == FAT_DTYPE_F16) launch_merge_q<fat::F16>(prm, a, D, mgrid, stream);
  else if (a->q_dtype == FAT_DTYPE_BF16) launch_merge_q<fat::BF16>(prm, a, D, mgrid, stream);
  else launch_merge_q<fat::F32>(prm, a, D, mgrid, stream);
  return fat_host::launch_status("decode_merge_kernel");
}

}  // namespace

namespace {

// The kernel that a decode launch runs on (all sizes positive, kv the cache's
// KvKind).
struct DecodeRoute {
  int rpl;       // rows that one 16-byte load per lane covers
  bool fast_ok;  // the VALU and MFMA kernels take the shape
  bool generic;  // they don't, or the generic kernel is asked for ...
  bool lane;     // ... but the VALU kernel's per-lane form takes it
  bool mfma;
  int HG;        // (query head, token) rows per workgroup
};

void decode_route(const fat_decode_args* a, int kv, DecodeRoute* r) {
  const int D = a->head_dim;
  const int T = a->q_len > 1 ? a->q_len : 1;
  const int group = a->num_heads / a->num_kv_heads;
  // The VALU and MFMA kernels take fp16/bf16 queries, head_dim 64 or 128 and
  // power-of-two pages of at least the rows one 16-byte load per lane covers
  // (their loads read one page id per load); the generic kernel takes the rest.
  r->rpl = (kv == fat::KV_SAME) ? (D == 128 ? 4 : 8) : (D == 128 ? 8 : 16);
  // They address K/V through 32-bit byte offsets from a page's base: strides
  // non-negative, a page below 4 GB, the rows of one 32-key block below 2 GB.
  const int64_t qeb = a->q_dtype == FAT_DTYPE_F32 ? 4 : 2;
  const int64_t eb = (kv == fat::KV_SAME) ? qeb : 1;
  auto fits32 = [&](int64_t sp, int64_t ss, int64_t sh) {
    return sp >= 0 && ss >= 0 && sh >= 0 && eb * sp < (int64_t(1) << 32) && eb * (32 * ss + D) < (int64_t(1) << 31);
  };
  const bool strides_ok = fits32(a->k_stride_page, a->k_stride_slot, a->k_stride_head) &&
                          fits32(a->v_stride_page, a->v_stride_slot, a->v_stride_head);
  r->fast_ok = a->q_dtype != FAT_DTYPE_F32 && (D == 64 || D == 128) && ilog2_exact(a->page_size) >= 0 &&
               a->page_size >= r->rpl && strides_ok;
  r->generic = a->kernel == FAT_KERNEL_DECODE_GENERIC || (a->kernel == FAT_KERNEL_AUTO && !r->fast_ok);
  // Of the shapes the fast kernels refuse, the VALU kernel's per-lane form
  // takes those it is built for, with 16-byte aligned queries and strides
  // that fit its 32-bit factors; the generic kernel keeps the rest.  A group
  // of more than 4 heads reads its K/V once per 4 heads, most of it from L2,
  // and is still the faster form (fp16 page 1, B32: 64/8 heads ctx 2000 223 ->
  // 90.6 us, 32/1 heads ctx 8000 262 -> 101 us; fp32 64/8 ctx 1000 123 -> 82.6).
  const uintptr_t q_align =
      (uintptr_t)a->q | (uintptr_t)(qeb * a->q_stride_b) | (uintptr_t)(qeb * a->q_stride_h);
  r->lane = r->generic && T == 1 && a->kernel == FAT_KERNEL_AUTO && lane_takes(a->q_dtype, kv, D) && strides_ok &&
            (q_align & 15) == 0;
  r->mfma = group >= fat::kDecMfmaMinGroup || (kv != fat::KV_SAME && FAT_DEC_MFMA_8BIT);
  if (a->kernel == FAT_KERNEL_DECODE_VALU || a->kernel == FAT_KERNEL_DECODE_MFMA)
    r->mfma = a->kernel == FAT_KERNEL_DECODE_MFMA;
  if (T > 1) r->mfma = true;  // only the MFMA kernel has per-token rows
  r->HG = r->lane      ? 4
          : r->generic ? (group < fat_host::kGenericHeads ? group : fat_host::kGenericHeads)
                       : (r->mfma ? 32 : (group >= 8 ? 8 : 4));
}

// KV heads whose rows of one token lie in one 128-byte line of K and of V.
int line_heads(const fat_decode_args* a, int eb) {
  const int n = 128 / (eb * a->head_dim);
  return n > 1 && a->num_kv_heads % n == 0 && a->k_stride_head == a->head_dim && a->v_stride_head == a->head_dim ? n
                                                                                                              : 1;
}

// K/V storage of a launch, or -1 where the types don't go together.
int kv_kind(const fat_decode_args* a) {
  if (a->kv_dtype == a->q_dtype) return fat::KV_SAME;
  if (a->q_dtype == FAT_DTYPE_F32) return -1;
  if (a->kv_dtype == FAT_DTYPE_I8) return fat::KV_I8;
  return a->kv_dtype == FAT_DTYPE_FP8E4M3 ? fat::KV_FP8 : -1;
}

// Rows of a workgroup of a balanced launch, or 0 when `a` can't run as one:
// its kernel, more rows than its merge takes, or more sequences than it keeps
// in LDS.
int balanced_rows(const fat_decode_args* a, int kv, const DecodeRoute& r) {
  const int rows = std::min(r.HG, a->num_heads / a->num_kv_heads * (a->q_len > 1 ? a->q_len : 1));
  if (!a->balanced || (r.generic && !r.lane) || rows > fat::kBalRows || a->batch > fat::kBalMaxSeqs) return 0;
  // Forms that are built: the VALU kernel's (4-head groups; per lane but for
  // 16-bit head_dim 256, which spills) and the MFMA kernel's for 8-bit caches
  // (16-bit ones spill, and their many rows merge slower than in a kernel of
  // its own: four tokens each, 16 sequences of 1000-7900, 53.7 us in equal
  // partitions, 58 balanced).
  if (r.lane) return kv == fat::KV_SAME && a->head_dim > 128 ? 0 : rows;
  if (r.mfma) return kv == fat::KV_SAME ? 0 : rows;
  return kv == fat::KV_SAME && r.HG == 4 ? rows : 0;
}

// Two 4-wave workgroups per CU: one finds its place, starts an item or merges
// while the other streams (256 of 8 waves: 2 % faster on the largest batches,
// 2-14 % slower on the others).
int balanced_groups(const fat_decode_args* a) { return a->balanced > 1 ? a->balanced : 512; }

// Its workspace: two partial rows (acc, m, l) per row and workgroup.
size_t balanced_bytes(const fat_decode_args* a, int rows) {
  return (size_t)balanced_groups(a) * 2 * rows * (a->head_dim + 2) * sizeof(float);
}

}  // namespace

extern "C" size_t fat_paged_decode_balanced_workspace_bytes(const fat_decode_args* a) {
  if (!a || a->batch <= 0 || a->num_heads <= 0 || a->num_kv_heads <= 0 || a->num_heads % a->num_kv_heads != 0 ||
      a->head_dim < 16 || a->page_size < 1 || a->balanced < 0 || a->balanced > 4096)
    return 0;
  const int kv = kv_kind(a);
  if (kv < 0) return 0;
  DecodeRoute r;
  decode_route(a, kv, &r);
  const int rows = balanced_rows(a, kv, r);
  return rows ? balanced_bytes(a, rows) : 0;
}

extern "C" size_t fat_paged_decode_workspace_bytes(int32_t batch, int32_t num_heads, int32_t head_dim,
                                                   int32_t split_k) {
  if (split_k <= 1 || batch <= 0 || num_heads <= 0 || head_dim <= 0) return 0;
  return (size_t)batch * num_heads * split_k * (head_dim + 2) * sizeof(float);
}

// One counter per (query row, head): at least one per (sequence, token
// group, head group) of any kernel's grid.
extern "C" size_t fat_paged_decode_counters_bytes(int32_t rows, int32_t num_heads) {
  if (rows <= 0 || num_heads <= 0) return 0;
  return (size_t)rows * num_heads * sizeof(int32_t);
}

extern "C" int fat_paged_decode(const fat_decode_args* a, void* stream_ptr) {
  fat_host::clear_error();
  if (!a) {
    fat_host::set_error("fat_paged_decode: args is NULL");
    return FAT_E_INVALID;
  }
  if (!a->q || !a->k_cache || !a->v_cache || !a->page_table || !a->seq_lens || !a->out) {
    fat_host::set_error("fat_paged_decode: a required pointer is NULL");
    return FAT_E_INVALID;
  }
  if (a->batch <= 0 || a->num_heads <= 0 || a->num_kv_heads <= 0 || a->num_pages <= 0 || a->max_pages <= 0) {
    fat_host::set_error("fat_paged_decode: batch, heads, num_pages and max_pages must be positive");
    return FAT_E_INVALID;
  }
  if (a->num_heads % a->num_kv_heads != 0) {
    fat_host::set_error("fat_paged_decode: num_heads %d must be divisible by num_kv_heads %d", a->num_heads,
                        a->num_kv_heads);
    return FAT_E_INVALID;
  }
  if (a->split_k < 1 || a->split_k > 64) {
    fat_host::set_error("fat_paged_decode: split_k must be in [1, 64], got %d", a->split_k);
    return FAT_E_INVALID;
  }
  if (a->q_dtype != FAT_DTYPE_F16 && a->q_dtype != FAT_DTYPE_BF16 && a->q_dtype != FAT_DTYPE_F32) {
    fat_host::set_error("fat_paged_decode: q_dtype must be fp16, bf16 or fp32");
    return FAT_E_UNSUPPORTED;
  }
  const int kv = kv_kind(a);
  if (kv < 0) {
    fat_host::set_error("fat_paged_decode: kv_dtype must equal q_dtype, or be int8/fp8e4m3 with fp16/bf16 queries");
    return FAT_E_UNSUPPORTED;
  }
  if (kv != fat::KV_SAME && (!a->k_scale || !a->v_scale)) {
    fat_host::set_error("fat_paged_decode: int8/fp8 K/V need k_scale and v_scale");
    return FAT_E_INVALID;
  }
  const int D = a->head_dim;
  if (D < 16 || D > 512 || (D & (D - 1)) != 0) {
    fat_host::set_error("fat_paged_decode: head_dim %d unsupported (a power of two from 16 to 512)", D);
    return FAT_E_UNSUPPORTED;
  }
  if (a->page_size < 1) {
    fat_host::set_error("fat_paged_decode: page_size must be positive, got %d", a->page_size);
    return FAT_E_INVALID;
  }
  const int log2P = ilog2_exact(a->page_size);
  if (a->waves_per_group != 0 && a->waves_per_group != 4 && a->waves_per_group != 8) {
    fat_host::set_error("fat_paged_decode: waves_per_group must be 0 (auto), 4 or 8, got %d", a->waves_per_group);
    return FAT_E_INVALID;
  }
  if (a->pages_per_split < 0) {
    fat_host::set_error("fat_paged_decode: pages_per_split must be >= 0, got %d", a->pages_per_split);
    return FAT_E_INVALID;
  }
  if (a->split_k > 1 && !a->workspace) {
    fat_host::set_error("fat_paged_decode: split_k > 1 needs a workspace");
    return FAT_E_INVALID;
  }
  if (a->balanced < 0 || a->balanced > 4096) {
    fat_host::set_error("fat_paged_decode: balanced must be in [0, 4096], got %d", a->balanced);
    return FAT_E_INVALID;
  }
  if ((uintptr_t)a->merge_counters & 3) {
    fat_host::set_error("fat_paged_decode: merge_counters must be 4-byte aligned");
    return FAT_E_INVALID;
  }
  if (a->workspace_bytes < 0) {
    fat_host::set_error("fat_paged_decode: workspace_bytes must be >= 0, got %lld", (long long)a->workspace_bytes);
    return FAT_E_INVALID;
  }
  if (a->q_len < 0 || a->q_len > 64) {
    fat_host::set_error("fat_paged_decode: q_len must be in [0, 64] (0 and 1 = one query per sequence), got %d",
                        a->q_len);
    return FAT_E_INVALID;
  }
  const int T = a->q_len > 1 ? a->q_len : 1;
  if (a->kernel != FAT_KERNEL_AUTO && a->kernel != FAT_KERNEL_DECODE_VALU && a->kernel != FAT_KERNEL_DECODE_MFMA &&
      a->kernel != FAT_KERNEL_DECODE_GENERIC) {
    fat_host::set_error("fat_paged_decode: kernel must be FAT_KERNEL_AUTO (0), _DECODE_VALU (1), _DECODE_MFMA (2) "
                        "or _DECODE_GENERIC (3), got %d", a->kernel);
    return FAT_E_INVALID;
  }
  if (a->kernel == FAT_KERNEL_DECODE_VALU && T > 1) {
    fat_host::set_error("fat_paged_decode: the VALU decode kernel takes one query per sequence (q_len %d)", T);
    return FAT_E_UNSUPPORTED;
  }
  DecodeRoute route;
  decode_route(a, kv, &route);
  const bool generic = route.generic, fast_ok = route.fast_ok;
  const int rpl = route.rpl;
  if (!generic && !fast_ok) {
    fat_host::set_error("fat_paged_decode: the %s decode kernel takes fp16/bf16 queries, head_dim 64 or 128, "
                        "power-of-two pages of at least %d rows and non-negative K/V strides with pages below "
                        "4 GB (page_size %d, head_dim %d); use FAT_KERNEL_AUTO or FAT_KERNEL_DECODE_GENERIC",
                        a->kernel == FAT_KERNEL_DECODE_VALU ? "VALU" : "MFMA", rpl, a->page_size, D);
    return FAT_E_UNSUPPORTED;
  }
  if (generic && T > 1) {
    fat_host::set_error("fat_paged_decode: multi-token decode (q_len %d) runs on the MFMA kernel, which takes "
                        "fp16/bf16, head_dim 64 or 128 and power-of-two pages of at least %d rows", T, rpl);
    return FAT_E_UNSUPPORTED;
  }
  // 16-byte alignment of every row start the kernels load.
  const int qeb = a->q_dtype == FAT_DTYPE_F32 ? 4 : 2;
  const int eb = (kv == fat::KV_SAME) ? qeb : 1;
  const uintptr_t q_align = generic ? 0
                                    : ((uintptr_t)a->q | (uintptr_t)(qeb * a->q_stride_b) |
                                       (uintptr_t)(qeb * a->q_stride_h) | (uintptr_t)(T > 1 ? qeb * a->q_stride_t : 0));
  const uintptr_t align_or = q_align | (uintptr_t)a->k_cache | (uintptr_t)a->v_cache |
                             (uintptr_t)(eb * a->k_stride_page) | (uintptr_t)(eb * a->k_stride_slot) |
                             (uintptr_t)(eb * a->k_stride_head) | (uintptr_t)(eb * a->v_stride_page) |
                             (uintptr_t)(eb * a->v_stride_slot) | (uintptr_t)(eb * a->v_stride_head);
  if (align_or & 15) {
    fat_host::set_error("fat_paged_decode: q/K/V base pointers and row strides must be 16-byte aligned");
    return FAT_E_INVALID;
  }

  const int group = a->num_heads / a->num_kv_heads;
  const bool lane = route.lane, use_mfma = route.mfma;
  if (!generic && !use_mfma && kv != fat::KV_SAME && group >= 8) {
    fat_host::set_error("fat_paged_decode: the VALU decode takes int8/fp8 caches for GQA groups below 8 "
                        "(group %d); use FAT_KERNEL_AUTO or FAT_KERNEL_DECODE_MFMA", group);
    return FAT_E_UNSUPPORTED;
  }
  const int HG = route.HG;
  const int hg_per_kv = (group * T + HG - 1) / HG;

  fat::DecodeParams prm{};
  prm.q = static_cast<const uint8_t*>(a->q);
  prm.k = static_cast<const uint8_t*>(a->k_cache);
  prm.v = static_cast<const uint8_t*>(a->v_cache);
  prm.ks = a->k_scale;
  prm.vs = a->v_scale;
  prm.pt = a->page_table;
  prm.lens = a->seq_lens;
  prm.out = static_cast<uint8_t*>(a->out);
  const size_t acc_elems = (size_t)a->batch * T * a->num_heads * a->split_k * D;
  prm.ws_acc = a->split_k > 1 ? static_cast<float*>(a->workspace) : nullptr;
  prm.ws_ml = a->split_k > 1 ? static_cast<float*>(a->workspace) + acc_elems : nullptr;
  prm.q_sb = a->q_stride_b;
  prm.q_sh = a->q_stride_h;
  prm.q_st = T > 1 ? a->q_stride_t : 0;
  prm.k_sp = a->k_stride_page;
  prm.k_ss = a->k_stride_slot;
  prm.k_sh = a->k_stride_head;
  prm.v_sp = a->v_stride_page;
  prm.v_ss = a->v_stride_slot;
  prm.v_sh = a->v_stride_head;
  prm.sc_sp = a->scale_stride_page;
  prm.sc_sh = a->scale_stride_head;
  prm.pt_sb = a->page_table_stride;
  prm.o_sb = a->out_stride_b;
  prm.o_sh = a->out_stride_h;
  prm.o_st = T > 1 ? a->out_stride_t : 0;
  prm.T = T;
  prm.H = a->num_heads;
  prm.Hkv = a->num_kv_heads;
  prm.group = group;
  prm.hg_per_kv = hg_per_kv;
  prm.P = a->page_size;
  prm.log2P = log2P;
  prm.invP = a->page_size > 1 ? (uint32_t)((uint64_t(1) << 32) / (uint32_t)a->page_size) : 0;
  prm.num_pages = a->num_pages;
  prm.max_pages = a->max_pages;
  prm.pps_fixed = a->pages_per_split;
  prm.scale_log2 = a->softmax_scale * fat::kLog2e;
  // Split-K merge inside the decode launch (VALU and MFMA kernels, split_k
  // <= 16) when the caller gives the counters and a workgroup's rows make at
  // most two output elements per thread: the last workgroup of a head group
  // merges alone, so wider groups (e.g. MQA's 32 heads) and more partitions
  // keep the merge kernel, which spreads the elements over many workgroups
  // (measured on MI355X: 32 partitions merged in the launch ran 1-11 %
  // slower, 16 and fewer 2-21 % faster).
  const int S = a->split_k;
  auto use_fused = [&](int rows_per_wg, int nw) {
    return S > 1 && S <= 16 && a->merge_counters != nullptr && rows_per_wg * D <= 2 * 64 * nw;
  };
  bool fused = false;
  prm.counters = nullptr;
  prm.smax = S <= 4 ? 4 : S <= 8 ? 8 : 16;

  hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
  const dim3 grid(a->split_k, a->num_kv_heads * hg_per_kv, a->batch);
  const int64_t wgs = (int64_t)grid.x * grid.y * grid.z;
  prm.share = wgs < (1LL << 31) ? hg_per_kv * line_heads(a, eb) : 1;
  const int64_t pages_per_wg =
      a->pages_per_split > 0 ? a->pages_per_split : ((int64_t)a->max_pages + a->split_k - 1) / a->split_k;
  const int bal_rows = a->workspace && a->merge_counters ? balanced_rows(a, kv, route) : 0;
  const size_t ws_need = bal_rows ? balanced_bytes(a, bal_rows)
                                  : fat_paged_decode_workspace_bytes(a->batch * T, a->num_heads, D, a->split_k);
  if (a->workspace_bytes > 0 && ws_need > (size_t)a->workspace_bytes) {
    fat_host::set_error("fat_paged_decode: this launch needs %zu bytes of workspace, the caller's holds %lld", ws_need,
                        (long long)a->workspace_bytes);
    return FAT_E_INVALID;
  }
  if (bal_rows) {
    const int groups = balanced_groups(a);
    prm.counters = a->merge_counters;
    prm.B = a->batch;
    prm.bal_rows = bal_rows;
    prm.ws_acc = static_cast<float*>(a->workspace);
    prm.ws_ml = prm.ws_acc + (size_t)groups * 2 * bal_rows * D;
    return fat_host::launch_decode_balanced(prm, a->q_dtype, kv, lane, D, groups, stream);
  }
  if (lane) {
    const int nw = a->waves_per_group ? a->waves_per_group
                                      : ((wgs < 2 * 256 || pages_per_wg * a->page_size >= 1024) ? 8 : 4);
    fused = use_fused(std::min(HG, group), nw);
    prm.counters = fused ? a->merge_counters : nullptr;
    const int rc = launch_lane(prm, a->q_dtype, kv, D, nw, grid, stream);
    if (rc != FAT_OK || a->split_k == 1 || fused) return rc;
    return launch_merge(prm, a, D, stream);
  }
  if (generic) {
    const int rc = fat_host::launch_decode_generic(prm, a->q_dtype, kv, D, HG, grid, stream);
    if (rc != FAT_OK || a->split_k == 1) return rc;
    return launch_merge(prm, a, D, stream);
  }
  if (use_mfma) {
    // 8 waves per workgroup pay off only when the grid leaves CUs short of
    // workgroups and each partition is long (>= 2048 keys, measured on
    // MI355X); short partitions finish sooner with 4.
    int nw = a->waves_per_group ? a->waves_per_group
                                : ((wgs < 2 * 256 && pages_per_wg * a->page_size >= 2048) ? 8 : 4);
    fused = use_fused(std::min(32, group * T), nw);
    prm.counters = fused ? a->merge_counters : nullptr;
    if (a->q_dtype == FAT_DTYPE_F16) launch_decode_mfma_q<fat::F16>(prm, kv, D, nw, grid, stream);
    else launch_decode_mfma_q<fat::BF16>(prm, kv, D, nw, grid, stream);
    const int rc = fat_host::launch_status("paged_decode_mfma_kernel");
    if (rc != FAT_OK || a->split_k == 1 || fused) return rc;
    return launch_merge(prm, a, D, stream);
  }
  // 8-wave workgroups keep more loads in flight per CU.  They pay off when
  // fewer than two 4-wave workgroups per CU leave the 256 CUs short of waves,
  // and in any grid when each partition is long (>= 1024 keys: +8-12 % at
  // B128, ctx 1024-16384, measured on MI355X); short partitions in big grids
  // finish sooner with 4.
  const int nw = a->waves_per_group ? a->waves_per_group
                                    : ((wgs < 2 * 256 || pages_per_wg * a->page_size >= 1024) ? 8 : 4);
  fused = use_fused(std::min(HG, group), nw);
  prm.counters = fused ? a->merge_counters : nullptr;
  int rc = (a->q_dtype == FAT_DTYPE_F16) ? launch_decode_q<fat::F16>(prm, kv, D, HG, nw, grid, stream)
                                         : launch_decode_q<fat::BF16>(prm, kv, D, HG, nw, grid, stream);
  if (rc != FAT_OK || a->split_k == 1 || fused) return rc;

  return launch_merge(prm, a, D, stream);
}

// ---------------------------------------------------------------------------
// Allocation-free decode: the split-K workspace lives in a file-scope device
// array instead of caller memory.  Every GPU the library runs on holds its
// own copy of `scratch` (kScratchBytes) until the process ends.  Its device
// address is looked up once per device with hipGetSymbolAddress (the array's
// name is only a host-side stand-in) and used for every launch after that.
// Nothing in it needs clearing: each partition of a launch writes its whole
// (acc, m, l) row before the merge reads it.  Two calls that overlap on one
// GPU (different streams) share the array and race.
// ---------------------------------------------------------------------------
namespace {

constexpr size_t kScratchBytes = FAT_DECODE_NOALLOC_MAX_WORKSPACE;
constexpr int kMaxDevices = 64;

__device__ __align__(256) uint8_t scratch[kScratchBytes];

std::once_flag g_scratch_once[kMaxDevices];
void* g_scratch_ptr[kMaxDevices];
hipError_t g_scratch_err[kMaxDevices];

}  // namespace

extern "C" int fat_paged_decode_noalloc(const fat_decode_args* a, void* stream) {
  fat_host::clear_error();
  if (!a) {
    fat_host::set_error("fat_paged_decode_noalloc: args is NULL");
    return FAT_E_INVALID;
  }
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    fat_host::set_error("fat_paged_decode_noalloc: no current HIP device (or device id >= %d)", kMaxDevices);
    return FAT_E_INVALID;
  }
  // The array is per device: a stream of another device would get this
  // device's address and fault or corrupt there.
  if (stream) {
    hipDevice_t sdev = -1;
    if (hipStreamGetDevice(static_cast<hipStream_t>(stream), &sdev) != hipSuccess || sdev != dev) {
      fat_host::set_error("fat_paged_decode_noalloc: the stream belongs to device %d, the current device is %d",
                          (int)sdev, dev);
      return FAT_E_INVALID;
    }
  }
  std::call_once(g_scratch_once[dev], [dev] {
    void* ptr = nullptr;
    g_scratch_err[dev] = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    g_scratch_ptr[dev] = g_scratch_err[dev] == hipSuccess ? ptr : nullptr;
  });
  if (g_scratch_err[dev] != hipSuccess || !g_scratch_ptr[dev]) {
    fat_host::set_error("fat_paged_decode_noalloc: hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                        hipGetErrorString(g_scratch_err[dev]));
    return FAT_E_LAUNCH;
  }
  if (a->batch <= 0 || a->num_heads <= 0 || a->head_dim <= 0 || a->split_k < 1 || a->q_len < 0) {
    return fat_paged_decode(a, stream);  // the regular entry reports the bad argument
  }
  const int64_t rows = (int64_t)a->batch * (a->q_len > 1 ? a->q_len : 1);
  const size_t need = a->split_k > 1 ? (size_t)rows * a->num_heads * a->split_k * (a->head_dim + 2) * sizeof(float)
                                     : 0;
  if (need > kScratchBytes) {
    fat_host::set_error("fat_paged_decode_noalloc: this launch needs %zu bytes of split-K workspace; the "
                        "allocation-free entry holds at most %zu (lower split_k, or use fat_paged_decode with a "
                        "workspace)", need, kScratchBytes);
    return FAT_E_INVALID;
  }
  fat_decode_args b = *a;
  b.workspace = need ? g_scratch_ptr[dev] : nullptr;
  b.workspace_bytes = (int64_t)kScratchBytes;
  b.merge_counters = nullptr;  // a second kernel merges: no state outside the scratch array
  const int rc = fat_paged_decode(&b, stream);
  if (rc != FAT_OK) {
    // Name this entry in the message the shared path set.
    char msg[480];
    snprintf(msg, sizeof(msg), "%s", fat_last_error());
    fat_host::set_error("fat_paged_decode_noalloc: %s", msg);
  }
  return rc;
}
