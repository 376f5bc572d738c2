// decode_kernels.h -- the VALU and MFMA decode kernels (see decode.hip for the
// design and for which launch runs which), and the split-K merges inside the
// decode launch.  Instantiated by decode.hip (one partition per workgroup)
// and decode_balanced.hip (equal shares of the batch per workgroup).
#pragma once

#include <limits.h>

#include <type_traits>

#include "decode_params.h"

namespace fat {


// Lazy rescale bound of both decode kernels (log2 units): m only moves when
// a block's or unit's max exceeds it by more than this; p then stays below
// 2^kDecLazy.
constexpr float kDecLazy = 8.0f;

// fp16/bf16 K/V with at least this many query heads per KV head use the MFMA
// decode (the `kernel` argument field overrides the choice).
constexpr int kDecMfmaMinGroup = 8;

// K/V rows are read once per launch: streaming (nontemporal) loads.
#ifndef FAT_DEC_NT
#define FAT_DEC_NT 1
#endif
// A wave-uniform word that the kernel does not write, read by the scalar unit
// (through the constant address space): the compiler does so by itself only
// where no store of the kernel can come first, which the loop of a balanced
// launch undoes (its page ids then came through vector loads and waited for
// the K/V loads ahead of them: B32 ctx 4096 126 us instead of 87).
template <typename T>
__device__ __forceinline__ T uniform_load(const T* ptr, int64_t i) {
  return ((const __attribute__((address_space(4))) T*)ptr)[i];
}

// 16 bytes of K or V at base + off through a raw buffer descriptor of range
// `bytes` (offsets at or past it read as zeros); base is wave-uniform (a
// page's row), off the lane's chunk.  Cache policy 2 is the nt (streaming)
// bit of gfx950 loads.
__device__ __forceinline__ u32x4 kv_buffer_load(const uint8_t* base, int bytes, uint32_t off) {
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, bytes, kBufFlags);
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, FAT_DEC_NT ? 2 : 0));
}
#ifndef FAT_DEC_MFMA_8BIT
#define FAT_DEC_MFMA_8BIT 1
#endif


// Lane geometry: a row of D elements is held by at most 16 lanes, in kNc
// 16-byte chunks each (chunk c + kLpr * j of lane c, so that a row's lanes
// read consecutive chunks).
template <typename QT, int KV, int D>
struct Geom {
  static constexpr int kElemBytes = (KV == KV_SAME) ? Elem<QT>::kBytes : 1;
  static constexpr int kEpc = 16 / kElemBytes;  // elements per chunk
  static constexpr int kNc = D / kEpc > 16 ? D / kEpc / 16 : 1;  // chunks per lane per row
  static constexpr int kEpl = kEpc * kNc;       // elements per lane per row
  static constexpr int kLpr = D / kEpl;         // lanes per row
  static constexpr int kRpl = 64 / kLpr;        // rows per load
  static constexpr int kNi16 = kRpl < 16 ? 16 / kRpl : 1;  // row groups per 16 tokens
  // Tokens per streamed unit: 16, or 32 or 64 when 16 tokens take only two
  // or one loads per lane for each of K and V (fp16/bf16 at head_dim 64 or
  // 32), so a wave keeps as many bytes in flight as at head_dim 128.
  static constexpr int kUnitLog2 = (KV == KV_SAME && kNi16 == 2) ? 5 : (KV == KV_SAME && kNi16 == 1) ? 6 : 4;
  static constexpr int kUnit = 1 << kUnitLog2;
  static constexpr int kNi = kUnit / kRpl;      // row groups per unit
  static_assert(kLpr == 4 || kLpr == 8 || kLpr == 16, "unsupported head_dim / element size");
};

// One transposing butterfly step on lane bit BIT: NCUR values -> NCUR/2.
template <int BIT, int NCUR>
__device__ __forceinline__ void tr_step(float* x, bool up) {
#pragma unroll
  for (int j = 0; j < NCUR / 2; ++j) {
    const float lo = x[j];
    const float hi = x[j + NCUR / 2];
    const float slo = lo + row_partner<BIT>(lo);
    const float shi = hi + row_partner<BIT>(hi);
    x[j] = up ? shi : slo;
  }
}

// Sum N per-lane partials over the LPR lanes of a row; afterwards lane c
// holds the full sums of values j = c * (N / LPR) + k, k < N / LPR.
template <int LPR, int N>
__device__ __forceinline__ void transpose_reduce(float* x, int c) {
  static_assert(N >= LPR, "need at least one value per lane");
  if constexpr (LPR >= 16) tr_step<8, N>(x, (c & 8) != 0);
  if constexpr (LPR >= 8) tr_step<4, N * 8 / LPR>(x, (c & 4) != 0);
  if constexpr (LPR >= 4) tr_step<2, N * 4 / LPR>(x, (c & 2) != 0);
  tr_step<1, N * 2 / LPR>(x, (c & 1) != 0);
}

// Registers holding one unit's K/V rows (and per-load scales for 8-bit K/V).
template <int NI, int NC>
struct UnitRegs {
  u32x4 k[NI * NC];
  u32x4 v[NI * NC];
  float ksc[NI];
  float vsc[NI];
};

// 16 bytes of int8 or OCP e4m3 K as their exact values in fp16 (8 packed
// pairs).  With fp16 queries both decode kernels stage K this way and apply
// k_scale to the fp32 scores, as the reference's quantised kernel does
// (kernels/decode.py:419-429: k = float(x) * k_scale, scores in fp32):
// 5 (int8) or 2 (fp8) instructions per 4 elements instead of 11 or 8 for
// round_to_fp16(float(x) * scale).  V keeps that per-element dequantisation:
// folding v_scale into P would round P after a scale that differs per page,
// and pages whose scales differ by 2^15 or more (two can share a 32-key
// block) would leave the smaller one's P in fp16's subnormal range.
template <int KV>
__device__ __forceinline__ void k8_exact_f16(const u32x4& raw, u32 (&out)[8]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (KV == KV_I8) {
      // fp16 bits 0x6400 | u are 1024 + u exactly (u = x + 128, the byte with
      // its sign bit flipped); adding -1152 leaves x.
      const u32 u = raw[j] ^ 0x80808080u;
      const f16x2 bias = {(f16)-1152.0f, (f16)-1152.0f};
      out[2 * j] = __builtin_bit_cast(
          u32, __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + bias);
      out[2 * j + 1] = __builtin_bit_cast(
          u32, __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + bias);
    } else {  // OCP e4m3 -> fp16 is exact
      out[2 * j] = __builtin_bit_cast(u32, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(raw[j], 1.0f, false));
      out[2 * j + 1] = __builtin_bit_cast(u32, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(raw[j], 1.0f, true));
    }
  }
}

// Page ids of the first unit of keys a wave reads (rows first_row + i * RPL
// of its partition, i < N), loaded at kernel start together with seq_len when
// the partition's first page does not depend on seq_len (partition 0, or
// fixed-size partitions): the first K/V loads then wait one memory latency
// after the launch instead of two.  The indices are clamped into the table
// row.  Two empty asm statements order the loads: the sequence index passes
// through one with the table indices (so the seq_len load issues no earlier
// than the id loads, not ahead of argument loads they wait for), and seq_len
// through one with the ids (so the ids are loaded before seq_len's first use
// instead of where they are used, after the wait for seq_len).  Neither is
// volatile or touches memory, so the loads, and later table reads, stay
// scalar loads.
template <int N, int RPL>
__device__ __forceinline__ int first_page_ids(int* pid, const int32_t* ptrow, const DecodeParams& p, int split,
                                              int first_row, int b, bool early) {
  if (!early) return p.lens[b];
  const int64_t pg0 = p.pps_fixed > 0 ? (int64_t)split * p.pps_fixed : 0;
  int64_t idx[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    idx[i] = min(pg0 + ((first_row + i * RPL) >> p.log2P), (int64_t)p.max_pages - 1);
    asm("" : "+s"(b) : "s"(idx[i]));
  }
  int seq_len = p.lens[b];
#pragma unroll
  for (int i = 0; i < N; ++i) pid[i] = ptrow[idx[i]];
#pragma unroll
  for (int i = 0; i < N; ++i) asm("" : "+s"(pid[i]), "+s"(seq_len));
  return seq_len;
}

// One output element of the split-K merge: row bh (its S partitions'
// (acc, m, l) in the workspace), head dim d, stored at element o of out.
// SMAX (a power of two >= S) fixes the trip count so the loops unroll:
// every partition's (m, l) and acc loads are issued before the first is used,
// one memory latency instead of one per partition.  Padded partitions
// (s >= S) re-read partition S - 1, so every address is inside the row, and
// are then given m = -inf (weight 0).
// COH: the rows were written by other workgroups of this launch with
// device-scope stores (ws_store); they are read with device-scope loads.
template <bool COH>
__device__ __forceinline__ float ws_load(const float* ptr) {
  if constexpr (COH) return __hip_atomic_load(ptr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return *ptr;
}
__device__ __forceinline__ void ws_store(float* ptr, float v, bool coh) {
  if (coh) __hip_atomic_store(ptr, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *ptr = v;
}

template <typename QT, int SMAX, bool COH = false>
__device__ __forceinline__ void merge_elem(const float* __restrict__ ws_acc, const float* __restrict__ ws_ml,
                                           int64_t bh, int d, int D, int S, uint8_t* out, int64_t o) {
  const float* ml = ws_ml + bh * S * 2;
  const float* acc = ws_acc + bh * S * D + d;
  float m[SMAX], l[SMAX], a[SMAX];
#pragma unroll
  for (int s = 0; s < SMAX; ++s) {
    const int sc = min(s, S - 1);
    m[s] = ws_load<COH>(ml + 2 * sc);
    l[s] = ws_load<COH>(ml + 2 * sc + 1);
    a[s] = ws_load<COH>(acc + (int64_t)sc * D);
  }
#pragma unroll
  for (int s = 0; s < SMAX; ++s) {
    if (s >= S) {
      m[s] = -INFINITY;
      l[s] = 0.f;
      a[s] = 0.f;
    }
  }
  float M = -INFINITY;
#pragma unroll
  for (int s = 0; s < SMAX; ++s) M = fmaxf(M, m[s]);
  float A = 0.f, L = 0.f;
  if (M != -INFINITY) {
#pragma unroll
    for (int s = 0; s < SMAX; ++s) {
      const float f = fast_exp2(m[s] - M);  // 0 for padded or empty partitions
      A = __builtin_fmaf(a[s], f, A);
      L = __builtin_fmaf(l[s], f, L);
    }
  }
  store_elem<QT>(out, o, L > 0.f ? A / L : 0.f);
}

// The merge of merge_in_launch, with merge_elem's arithmetic: per row j (one
// thread each) M = max_s m_s, the weights f_s = 2^(m_s - M) (0 for padded
// partitions) and L = sum_s l_s f_s in partition order, kept in LDS; per
// output element A = sum_s acc_s f_s in partition order and A / L.  A
// thread takes at most two elements (the host fuses the merge only then)
// and issues their partial sums' loads together with its row's (m, l), so
// the merge waits for one memory latency.
template <typename QT, int D, int SMAX, typename RowOf>
__device__ __forceinline__ void merge_rows(const DecodeParams& p, int S, int nrows, RowOf row_of, float* s_f,
                                           float* s_l) {
  const int n = nrows * D;
  const int e0 = threadIdx.x, e1 = threadIdx.x + blockDim.x;  // this thread's elements (if < n)
  float a0[SMAX], a1[SMAX];
  int64_t o0 = 0, o1 = 0;
  auto load_acc = [&](int e, float (&a)[SMAX], int64_t& o) {
    const int j = e / D;
    const int d = e - j * D;
    int64_t bh;
    row_of(j, bh, o);
    o += d;
    const float* acc = p.ws_acc + bh * S * D + d;
#pragma unroll
    for (int s = 0; s < SMAX; ++s) a[s] = s < S ? ws_load<true>(acc + (int64_t)s * D) : 0.f;
  };
  if (e0 < n) load_acc(e0, a0, o0);
  if (e1 < n) load_acc(e1, a1, o1);
  if (threadIdx.x < nrows) {
    const int j = threadIdx.x;
    int64_t bh, o;
    row_of(j, bh, o);
    const float* ml = p.ws_ml + bh * S * 2;
    float m[SMAX], l[SMAX];
#pragma unroll
    for (int s = 0; s < SMAX; ++s) {
      const int sc = min(s, S - 1);
      m[s] = ws_load<true>(ml + 2 * sc);
      l[s] = ws_load<true>(ml + 2 * sc + 1);
    }
#pragma unroll
    for (int s = 0; s < SMAX; ++s) {
      if (s >= S) {
        m[s] = -INFINITY;
        l[s] = 0.f;
      }
    }
    float M = -INFINITY;
#pragma unroll
    for (int s = 0; s < SMAX; ++s) M = fmaxf(M, m[s]);
    float L = 0.f;
#pragma unroll
    for (int s = 0; s < SMAX; ++s) {
      const float f = M != -INFINITY ? fast_exp2(m[s] - M) : 0.f;
      s_f[j * SMAX + s] = f;
      L = __builtin_fmaf(l[s], f, L);
    }
    s_l[j] = M != -INFINITY ? L : -1.f;  // -1: no partition saw a key (output 0, as merge_elem)
  }
  __syncthreads();
  auto finish = [&](int e, const float (&a)[SMAX], int64_t o) {
    const int j = e / D;
    const float L = s_l[j];
    float A = 0.f;
    if (L >= 0.f) {
#pragma unroll
      for (int s = 0; s < SMAX; ++s) A = __builtin_fmaf(a[s], s_f[j * SMAX + s], A);
    }
    store_elem<QT>(p.out, o, L > 0.f ? A / L : 0.f);
  };
  if (e0 < n) finish(e0, a0, o0);
  if (e1 < n) finish(e1, a1, o1);
}

// The sequence, head group and partition of this workgroup: its place in the
// grid, or (share > 1) so that `share` consecutive head groups of a partition
// run on one XCD and close in time.  Workgroups go to the 8 XCDs in turn by
// their linear id, so workgroups 8 apart share an L2: 8 units of `share` head
// groups take each 8 * share ids, what remains of the grid the rest in order.
// The head groups' loads of the same lines then meet in that L2 instead of
// each going to memory (40 sequences of 8611 tokens, 16/8 heads, an int8 cache
// at head_dim 64, 7 partitions 127.6 -> 90.9 us; 54 of 1950, 32/1 heads, bf16,
// pages of one token, 8 head groups, 5 partitions 87.9 -> 55.8; fp32, 32/1
// heads, 16 of 1000-4000 60.9 -> 39.1.  A number of partitions that 8 divides
// did so by chance).
__device__ __forceinline__ void partition_item(const DecodeParams& p, int& b, int& y, int& split) {
  b = blockIdx.z;
  y = blockIdx.y;
  split = blockIdx.x;
  if (p.share == 1) return;
  const unsigned n = (unsigned)p.share, S = gridDim.x, units_y = gridDim.y / n;
  const unsigned id = split + S * (y + gridDim.y * b);
  const unsigned whole = units_y * S * gridDim.z / 8 * 8;  // units that go to the XCDs in rounds of 8
  unsigned unit, k;
  if (id < whole * n) {
    const unsigned round = id / (8 * n), r = id - round * 8 * n;
    unit = round * 8 + r % 8;
    k = r / 8;
  } else {
    unit = whole + (id - whole * n) / n;
    k = (id - whole * n) % n;
  }
  const unsigned row = unit / S;
  split = unit - row * S;
  b = row / units_y;
  y = (row - b * units_y) * n + k;
}

// Split-K merge inside the decode launch (p.counters set).  Every thread has
// written its part of this workgroup's (acc, m, l) rows with device-scope
// stores (ws_store, global_store ... sc1: written through to the level all
// XCDs share); each wave waits until its stores have completed there
// (vmcnt(0)), then the workgroup counts itself in on its (sequence, head
// group) counter with a device-scope atomic.  The workgroup that brings the
// count to S has therefore seen every other partition's count, each issued
// after that partition's rows were complete at the shared level; it reads
// them with device-scope loads (global_load ... sc1), merges them and puts
// the counter back to zero for the next launch.  The ordering rests on
// those gfx950 completion rules, not on release/acquire operations: an
// agent-scope release would write back the whole L2 of the XCD
// (buffer_wbl2), which measured 7-16 % slower on 8-sequence split
// launches.  No workgroup waits for another.
template <typename QT, int D, typename RowOf>
__device__ __forceinline__ void merge_in_launch(const DecodeParams& p, int S, int item, int nrows, RowOf row_of) {
  __shared__ int s_last;
  __shared__ float s_f[32 * 16];  // merge weights of up to 32 rows x 16 partitions
  __shared__ float s_l[32];
  __atomic_signal_fence(__ATOMIC_SEQ_CST);  // keep the row stores before the wait
  __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0): this wave's row stores are complete
  __syncthreads();
  int* const cnt = p.counters + item;
  if (threadIdx.x == 0) {
    const int prev = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = prev == S - 1;
  }
  __syncthreads();
  if (!s_last) return;
  switch (p.smax) {
    case 4: merge_rows<QT, D, 4>(p, S, nrows, row_of, s_f, s_l); break;
    case 8: merge_rows<QT, D, 8>(p, S, nrows, row_of, s_f, s_l); break;
    default: merge_rows<QT, D, 16>(p, S, nrows, row_of, s_f, s_l); break;
  }
  if (threadIdx.x == 0) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------
// Balanced launches (BAL instantiations): the batch's work is cut into blocks
// of 2^kWB tokens of one (sequence, head group) item, the items lie one behind
// the other (sequence-major), and each of the launch's W workgroups takes an
// equal run of blocks, which may end one item, hold some and begin another.
// The lengths are read on the device, so a launch prepared once stays
// balanced as they change.  An item that one workgroup holds alone goes
// straight to the output; of the others each workgroup writes a partial
// (acc, m, l), at most two of them (the item its run begins in the middle of,
// slot 0, and the one it leaves unfinished, slot 1), and the last of an
// item's workgroups to arrive merges them in order (as merge_in_launch does,
// with the same ordering rules).
//
// Why: partitions of a ragged batch, whether of one size or so many per
// sequence, leave the last workgroups of the grid running while others are
// done, and the more partitions, the more of them are all start-up and merge.
// 512 workgroups of four waves (768-2048: level to 20 % slower) against the
// best partitions: 64 sequences of 500-16000 tokens, 32/8 heads, head_dim 128,
// on an fp8 cache 151 -> 130.5 us (534 MB, 4.1 TB/s), on a bf16 one 228 ->
// 201, 32 of 500-4000 with pages of one token 54.5 -> 49.5, one of 100000 and
// 63 of 200 in fp16 109 -> 93.  A run counts an item's tokens and not what an
// item costs besides, so it loses where a batch holds many very short ones
// (256 log-uniform in [16, 8192], head_dim 64, 161 -> 208).
// ---------------------------------------------------------------------------

// s_cum[b] = blocks of a head group's items over the sequences before b, for
// b = 0 .. B (a sequence without tokens still has one, empty, block: its
// zeros are written there).  Every thread calls it; it ends in a barrier.
template <int NT, int WB>
__device__ __forceinline__ void bal_prefix(const DecodeParams& p, int* s_cum, int* s_w) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int64_t cap = min((int64_t)p.max_pages * p.P, (int64_t)INT_MAX);
  int carry = 0;
  if (tid == 0) s_cum[0] = 0;
  for (int base = 0; base < p.B; base += NT) {
    const int i = base + tid;
    int x = 0;
    if (i < p.B) {
      const int len = (int)min((int64_t)p.lens[i], cap);
      x = len > 0 ? ((len - 1) >> WB) + 1 : 1;
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(x, off);
      x += lane >= off ? y : 0;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    int total = 0, before = carry;
#pragma unroll
    for (int k = 0; k < NT / 64; ++k) {
      before += k < wave ? s_w[k] : 0;
      total += s_w[k];
    }
    if (i < p.B) s_cum[i + 1] = before + x;
    carry += total;
    __syncthreads();
  }
}

// The sequence whose blocks hold block q of a head group's row of items.
__device__ __forceinline__ int bal_sequence(const int* s_cum, int B, int q) {
  int lo = 0, hi = B;  // s_cum[lo] <= q < s_cum[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (s_cum[mid] <= q) lo = mid;
    else hi = mid;
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

// One workgroup's run of blocks and how the items in it are shared.
struct BalRun {
  long long U, W;  // blocks of the launch, workgroups that take some
  // The workgroup that holds block x: the largest w with floor(w U / W) <= x.
  __device__ __forceinline__ int owner(long long x) const { return (int)(((x + 1) * W - 1) / U); }
  __device__ __forceinline__ int begin(int w) const { return (int)(w * U / W); }
};

__device__ __forceinline__ const float* bal_acc(const DecodeParams& p, int w, int slot, int row, int D) {
  return p.ws_acc + (((int64_t)w * 2 + slot) * p.bal_rows + row) * D;
}
__device__ __forceinline__ const float* bal_ml(const DecodeParams& p, int w, int slot, int row) {
  return p.ws_ml + (((int64_t)w * 2 + slot) * p.bal_rows + row) * 2;
}

// Counts this workgroup's partial of an item in; the last of the item's n
// workgroups (w_first ..) merges its nrows rows: M = max m, weights 2^(m - M),
// O = sum acc f / sum l f over the workgroups in order, 64 of them at a time.
// s_f: kBalRows x 64 floats of LDS, s_ml: kBalRows x 2.
template <typename QT, int D, int NT, typename OutOf>
__device__ __forceinline__ void bal_merge(const DecodeParams& p, int item, int w_first, int n, int nrows, OutOf out_of,
                                          float* s_f, float* s_ml) {
  __shared__ int s_last;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  __atomic_signal_fence(__ATOMIC_SEQ_CST);  // keep the partial's stores before the wait
  __builtin_amdgcn_s_waitcnt(0x0F70);       // vmcnt(0): this wave's stores are complete
  __syncthreads();
  if (tid == 0)
    s_last = __hip_atomic_fetch_add(p.counters + item, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
  __syncthreads();
  if (!s_last) return;
  // Row maxima, and the first 64 workgroups' weights and sums.
  for (int j = wave; j < nrows; j += NT / 64) {
    float M = -INFINITY, m0 = -INFINITY, l0 = 0.f;
    for (int s = lane; s < n; s += 64) {
      const float* ml = bal_ml(p, w_first + s, s == 0 ? 1 : 0, j);
      const float m = ws_load<true>(ml);
      if (s == lane) {
        m0 = m;
        l0 = ws_load<true>(ml + 1);
      }
      M = fmaxf(M, m);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) M = fmaxf(M, __shfl_xor(M, off));
    const float f = M != -INFINITY ? fast_exp2(m0 - M) : 0.f;
    float L = l0 * f;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) L += __shfl_xor(L, off);
    s_f[j * 64 + lane] = f;
    if (lane == 0) {
      s_ml[2 * j] = M;
      s_ml[2 * j + 1] = L;
    }
  }
  __syncthreads();
  constexpr int KM = (kBalRows * D / 2 + NT - 1) / NT;  // pairs of outputs per thread
  float a0[KM], a1[KM];
#pragma unroll
  for (int k = 0; k < KM; ++k) a0[k] = a1[k] = 0.f;
  for (int base = 0; base < n; base += 64) {
    if (base > 0) {
      __syncthreads();  // the previous weights are read
      for (int j = wave; j < nrows; j += NT / 64) {
        const float M = s_ml[2 * j];
        float f = 0.f, l = 0.f;
        if (base + lane < n && M != -INFINITY) {
          const float* ml = bal_ml(p, w_first + base + lane, 0, j);
          f = fast_exp2(ws_load<true>(ml) - M);
          l = ws_load<true>(ml + 1);
        }
        float L = l * f;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) L += __shfl_xor(L, off);
        s_f[j * 64 + lane] = f;
        if (lane == 0) s_ml[2 * j + 1] += L;
      }
      __syncthreads();
    }
    const int cn = min(64, n - base);
#pragma unroll
    for (int k = 0; k < KM; ++k) {
      const int e = 2 * (tid + k * NT);
      const int j = e / D;
      if (j >= nrows) continue;
      for (int s0 = 0; s0 < cn; s0 += 16) {
        float x0[16], x1[16];
#pragma unroll
        for (int s = 0; s < 16; ++s) {
          const int w = base + min(s0 + s, cn - 1);  // past the end: the last one again, weight 0 below
          const uint64_t* ptr = reinterpret_cast<const uint64_t*>(bal_acc(p, w_first + w, w == 0 ? 1 : 0, j, D) + e % D);
          const uint64_t v = __hip_atomic_load(ptr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          x0[s] = as_f32((u32)v);
          x1[s] = as_f32((u32)(v >> 32));
        }
#pragma unroll
        for (int s = 0; s < 16; ++s) {
          const float f = s0 + s < cn ? s_f[j * 64 + s0 + s] : 0.f;
          a0[k] = __builtin_fmaf(x0[s], f, a0[k]);
          a1[k] = __builtin_fmaf(x1[s], f, a1[k]);
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < KM; ++k) {
    const int e = 2 * (tid + k * NT);
    const int j = e / D;
    if (j >= nrows) continue;
    const float L = s_ml[2 * j + 1];
    const int64_t o = out_of(j) + e % D;
    store_elem<QT>(p.out, o, L > 0.f ? a0[k] / L : 0.f);
    store_elem<QT>(p.out, o + 1, L > 0.f ? a1[k] / L : 0.f);
  }
  if (tid == 0) __hip_atomic_store(p.counters + item, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The kernel's arguments, loaded again from the kernel argument segment: kept
// over the loop of bal_run they would take more scalar registers than there
// are (30-75 spilled).
__device__ __forceinline__ DecodeParams reload_params() {
  typedef const __attribute__((address_space(4))) u32* words;
  words k = (words)__builtin_amdgcn_kernarg_segment_ptr();
  __asm__ volatile("" : "+s"(k));
  struct Raw {
    u32 w[sizeof(DecodeParams) / 4];
  } raw;
#pragma unroll
  for (unsigned i = 0; i < sizeof(DecodeParams) / 4; ++i) raw.w[i] = k[i];
  return __builtin_bit_cast(DecodeParams, raw);
}

// Runs segment(p, b, y, t_begin, t_end, slot, item, w_first, n) for every part of
// an item in this workgroup's run: tokens [t_begin, t_end) of sequence b and
// head group y; slot -1: the whole item, else the partial's slot and the
// item's n workgroups from w_first on.
template <int NT, int WB, typename Segment>
__device__ __forceinline__ void bal_run(const DecodeParams& args, Segment segment) {
  __shared__ int s_cum[kBalMaxSeqs + 1];
  __shared__ int s_w[NT / 64];
  bal_prefix<NT, WB>(args, s_cum, s_w);
  const int w = blockIdx.x;
  int x, x1;
  {
    BalRun run;
    run.U = (long long)__builtin_amdgcn_readfirstlane(s_cum[args.B]) * (args.Hkv * args.hg_per_kv);
    run.W = min((long long)gridDim.x, run.U);
    if (w >= run.W) return;
    x1 = run.begin(w + 1);
    x = run.begin(w);
  }
  while (x < x1) {
    const DecodeParams p = reload_params();
    const int G = p.Hkv * p.hg_per_kv;
    const int64_t cap = min((int64_t)p.max_pages * p.P, (int64_t)INT_MAX);
    BalRun run;
    run.U = (long long)__builtin_amdgcn_readfirstlane(s_cum[p.B]) * G;
    run.W = min((long long)gridDim.x, run.U);
    const int b = bal_sequence(s_cum, p.B, x / G);
    const int before = __builtin_amdgcn_readfirstlane(s_cum[b]);
    const int nb = __builtin_amdgcn_readfirstlane(s_cum[b + 1]) - before;  // blocks of the item
    const int r = x - before * G;
    const int y = r / nb;
    const int blk = r - y * nb;
    const int take = min(nb - blk, x1 - x);
    const int len = (int)max((int64_t)0, min((int64_t)uniform_load(p.lens, b), cap));
    const int t_begin = blk << WB;
    const int t_end = min((int64_t)len, (int64_t)(blk + take) << WB);
    const bool whole = take == nb;
    const int first = x - blk;  // the item's first block
    const int w_first = whole ? w : run.owner(first);
    const int n = whole ? 1 : run.owner(first + nb - 1) - w_first + 1;
    segment(p, b, y, t_begin, t_end, whole ? -1 : (blk > 0 ? 0 : 1), b * G + y, w_first, n);
    x += take;
    if (x < x1) __syncthreads();  // the segment's LDS is free for the next one
  }
}

// LANE: K/V rows are addressed per lane (its own page id, a 64-bit address)
// instead of per load, for pages that one load can straddle: page sizes below
// RPL rows or not a power of two.  It also takes fp32 caches and head_dim 32
// and 256, whatever the page size.  HBM-bound like the per-load form; a
// lane's page ids are loaded one unit ahead of the rows they address (a
// vector load, the 16 lanes of a row reading one word), so a unit's K/V loads
// do not wait for them.  Against the LDS-tiled generic kernel that took these
// shapes before (three workgroup barriers per 32 tokens), B32 with 32/8
// heads: fp16 D128 page 1 ctx 2000 178 -> 46.5 us (5.65 TB/s), fp16 D256
// page 16 ctx 1000 193 -> 45.8 us (5.7 TB/s), its int8 / fp8 205 -> 36.7 and
// 202 -> 34.5 us, fp32 D128 page 16 ctx 1000 98 -> 43.3 us (6.1 TB/s).
template <typename QT, int KV, int D, int HG, int NW, bool LANE = false, bool BAL = false>
__global__ __launch_bounds__(NW * 64) void paged_decode_kernel(const DecodeParams p) {
  using Gm = Geom<QT, KV, D>;
  constexpr int EPL = Gm::kEpl, LPR = Gm::kLpr, RPL = Gm::kRpl, NI = Gm::kNi, NC = Gm::kNc, EPC = Gm::kEpc;
  constexpr bool F32Q = std::is_same<QT, F32>::value;
  static_assert(LANE || (NC == 1 && !F32Q), "the per-load form takes one 16-bit or 8-bit chunk per lane");
  constexpr int NV = NI * HG;       // per-lane partial scores before the reduction
  constexpr int NPL = NV / LPR;     // scores per lane after it
  constexpr int VPH = NPL < NI ? NPL : NI;  // scores per lane per head
  constexpr int HPL = NPL / VPH;            // heads per lane
  constexpr int LPH = NI / VPH;             // lanes per head inside a row
  constexpr int QW = F32Q ? EPL : EPL / 2;  // q dwords per head per lane (packed pairs, or fp32)
  constexpr int QWC = QW / NC;              // of which per chunk
  static_assert(HG % 4 == 0, "HG must be a multiple of 4");

  __shared__ float s_p[NW][RPL][NV];
  __shared__ float s_alpha[NW][HG];
  __shared__ float s_red[NW][HG][D];
  __shared__ float s_ml[NW][HG][2];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane / LPR;
  const int c = lane % LPR;

  // One partition (or, BAL, one segment: tokens [seg_begin, seg_end)) of
  // sequence b and head group y: the kernel's body, to "// segment".
  auto segment = [&](const DecodeParams& p, const int b, const int y, const int split, const int S, const int seg_begin, const int seg_end,
                     const int slot, const int item, const int w_first, const int n_parts)
      __attribute__((always_inline)) {
  const int sub = y % p.hg_per_kv;
  const int kvh = y / p.hg_per_kv;
  const int head0 = kvh * p.group + sub * HG;
  const int nvalid = min(HG, p.group - sub * HG);

  // Page ids of this wave's first unit, read together with seq_len when
  // `early` (first_page_ids).
  constexpr int UL = Gm::kUnitLog2;
  const int32_t* ptrow = p.pt + (int64_t)b * p.pt_sb;
  const bool early = !BAL && (split == 0 || p.pps_fixed > 0);
  // LANE: this lane's page ids and slots of the unit that the next fetch
  // reads.  Rows before `end` (INT_MAX: not clamped) look up their own token,
  // later ones end - 1; table column and page id are clamped, so every
  // address lies in the pool.
  int lane_pid[NI], lane_slot[NI];
  auto lookup = [&](int first_tok, int end) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const uint32_t tok = (uint32_t)min(first_tok + i * RPL + r, end - 1);
      uint32_t lp;
      if (p.log2P >= 0) {
        lp = tok >> p.log2P;
      } else {  // floor(tok / P): the high product is it or one less
        lp = __umulhi(tok, p.invP);
        lp += tok - lp * (uint32_t)p.P >= (uint32_t)p.P ? 1u : 0u;
      }
      lane_slot[i] = (int)(tok - lp * (uint32_t)p.P);
      lane_pid[i] = ptrow[min((int)lp, p.max_pages - 1)];
    }
  };
  // Partition of this sequence's pages (decode.py:271-276 semantics).
  int first_pid[NI];
  int t_begin, t_end;
  if constexpr (BAL) {
    t_begin = seg_begin;
    t_end = seg_end;
  } else if constexpr (LANE) {
    // Fixed-size partitions and partition 0 begin at a page that does not
    // depend on seq_len (a begin past the table is clamped by the lookup).
    const int64_t cap = (int64_t)p.max_pages * p.P;
    if (early) lookup((int)min((int64_t)split * p.pps_fixed * p.P, min(cap, (int64_t)1 << 30)) + (w << UL), INT_MAX);
    const int seq_len = (int)max((int64_t)0, min((int64_t)p.lens[b], cap));
    const int np = (int)(((int64_t)seq_len + p.P - 1) / p.P);
    const int pps = p.pps_fixed > 0 ? p.pps_fixed : (np + S - 1) / S;
    const int pb = (int)min((int64_t)np, (int64_t)split * pps);
    const int pe = split == S - 1 ? np : (int)min((int64_t)np, (int64_t)pb + pps);
    t_begin = pb * p.P;
    t_end = (int)min((int64_t)seq_len, (int64_t)pe * p.P);
  } else {
    int seq_len = first_page_ids<NI, RPL>(first_pid, ptrow, p, split, w << UL, b, early);
    seq_len = max(0, min(seq_len, p.max_pages << p.log2P));
    const int np = (seq_len + p.P - 1) >> p.log2P;
    const int pps = p.pps_fixed > 0 ? p.pps_fixed : (np + S - 1) / S;
    const int pb = split * pps;
    const int pe = split == S - 1 ? np : min(np, pb + pps);
    t_begin = pb << p.log2P;
    t_end = min(seq_len, pe << p.log2P);
  }
  const int n_units = t_end > t_begin ? (t_end - t_begin + Gm::kUnit - 1) >> UL : 0;

  // q for the HG heads, packed pairs of QT or fp32 (padded heads reuse head0).
  u32 qv[HG][QW];
#pragma unroll
  for (int g = 0; g < HG; ++g) {
    const int h = head0 + (g < nvalid ? g : 0);
#pragma unroll
    for (int j = 0; j < QW / 4; ++j) {
      // dword 4 j of the lane: chunk 4 j / QWC, 16 bytes 4 j % QWC / 4 of its q dwords
      const int d = EPC * (c + LPR * (4 * j / QWC)) + (4 * j % QWC) * (F32Q ? 1 : 2);
      const u32x4 t = *reinterpret_cast<const u32x4*>(p.q + Elem<QT>::kBytes * (b * p.q_sb + h * p.q_sh + d));
      qv[g][4 * j + 0] = t[0];
      qv[g][4 * j + 1] = t[1];
      qv[g][4 * j + 2] = t[2];
      qv[g][4 * j + 3] = t[3];
    }
  }

  constexpr int EB = Gm::kElemBytes;
  // Load i of a unit covers rows rs .. rs + RPL - 1 of one page (page_size
  // >= RPL, rs a multiple of RPL): its address is wave-uniform (page id,
  // slot and KV head on the scalar unit, in a buffer descriptor) plus this
  // lane's loop-invariant offset (row r, chunk c).  The descriptor's range
  // ends with the partition's last row, so rows past t_end (and loads wholly
  // past it) read as zeros: their scores are masked, and zero V rows keep
  // p * v = 0.
  // Byte strides (the host keeps a page below 4 GB and RPL rows below 2 GB).
  const uint8_t* const kh = p.k + (int64_t)EB * kvh * p.k_sh;  // this KV head's slice of page 0
  const uint8_t* const vh = p.v + (int64_t)EB * kvh * p.v_sh;
  const uint32_t kpage = (uint32_t)(EB * p.k_sp), vpage = (uint32_t)(EB * p.v_sp);
  const uint32_t krow = (uint32_t)(EB * p.k_ss), vrow = (uint32_t)(EB * p.v_ss);
  const uint32_t lane_k = r * krow + EB * EPL * c;
  const uint32_t lane_v = r * vrow + EB * EPL * c;

  // first: u is this wave's first unit (first_pid holds its page ids).
  auto fetch = [&](UnitRegs<NI, NC>& R, int u, bool first) __attribute__((always_inline)) {
    const int base = t_begin + (u << UL);
    if constexpr (LANE) {
      int phys[NI], slot[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        phys[i] = min(max(lane_pid[i], 0), p.num_pages - 1);
        slot[i] = lane_slot[i];
      }
      // The next unit's ids go out ahead of this unit's rows: loads return in
      // order, so waiting for them leaves the rows in flight.
      lookup(base + (NW << UL), t_end);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const uint8_t* kp = kh + ((uint64_t)(uint32_t)phys[i] * kpage + (uint64_t)(uint32_t)slot[i] * krow + 16 * c);
        const uint8_t* vp = vh + ((uint64_t)(uint32_t)phys[i] * vpage + (uint64_t)(uint32_t)slot[i] * vrow + 16 * c);
#pragma unroll
        for (int j = 0; j < NC; ++j) {
          R.k[i * NC + j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kp + 16 * LPR * j));
          R.v[i * NC + j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vp + 16 * LPR * j));
        }
        if constexpr (KV != KV_SAME) {
          R.ksc[i] = p.ks[(int64_t)phys[i] * p.sc_sp + (int64_t)kvh * p.sc_sh];
          R.vsc[i] = p.vs[(int64_t)phys[i] * p.sc_sp + (int64_t)kvh * p.sc_sh];
        }
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int rs = base + i * RPL;
      const int nrow = min(t_end - rs, RPL);  // rows of this load in the partition
      // The table is read without a branch (at most its last entry) so that
      // a unit's page-id loads issue together; a load wholly past t_end reads
      // nothing (range 0).  8-bit caches: it names the page of a row before
      // t_end, since the scales of a column that the sequence doesn't use can
      // be anything, and 0 * NaN would reach acc.
      int phys;
      if constexpr (KV == KV_SAME)
        phys = first && early ? first_pid[i] : uniform_load(ptrow, min(rs >> p.log2P, p.max_pages - 1));
      else
        phys = first && early ? (nrow > 0 ? first_pid[i] : first_pid[0])
                              : uniform_load(ptrow, min(rs, t_end - 1) >> p.log2P);
      phys = __builtin_amdgcn_readfirstlane(min(max(phys, 0), p.num_pages - 1));
      const uint32_t slot0 = (uint32_t)(rs & (p.P - 1));
      // range: the load's rows inside the partition, each up to its head slice's end
      const int nk = nrow > 0 ? (int)((uint32_t)(nrow - 1) * krow + EB * D) : 0;
      const int nv = nrow > 0 ? (int)((uint32_t)(nrow - 1) * vrow + EB * D) : 0;
      R.k[i] = kv_buffer_load(kh + (uint64_t)(uint32_t)phys * kpage + slot0 * krow, nk, lane_k);
      R.v[i] = kv_buffer_load(vh + (uint64_t)(uint32_t)phys * vpage + slot0 * vrow, nv, lane_v);
      if constexpr (KV != KV_SAME) {
        R.ksc[i] = uniform_load(p.ks, (int64_t)phys * p.sc_sp + (int64_t)kvh * p.sc_sh);
        R.vsc[i] = uniform_load(p.vs, (int64_t)phys * p.sc_sp + (int64_t)kvh * p.sc_sh);
      }
    }
  };

  // FOLD: exact 8-bit K and k_scale on the scores (k8_exact_f16).
  constexpr bool FOLD = KV != KV_SAME && std::is_same<QT, F16>::value;
  // Dequantise 16 bytes of 8-bit K/V into EPL/2 packed QT pairs:
  // round_to_QT(float(x) * scale).
  auto deq_pairs = [&](const u32x4& raw, float sc, u32* out) {
    const float nb = -128.0f * sc;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float f[4];
      if constexpr (KV == KV_I8) {
        i8x4_biased(raw[j], f);
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = __builtin_fmaf(f[e], sc, nb);
      } else {
        fp8x4(raw[j], f);
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = f[e] * sc;
      }
      if constexpr (!F32Q) {
        out[2 * j + 0] = Pair<QT>::pack(f[0], f[1]);
        out[2 * j + 1] = Pair<QT>::pack(f[2], f[3]);
      }
    }
  };

  // Finite, so that a wave whose first units hold only scores of -inf gets
  // p = 2^(-inf) = 0 for them, and not the NaN of -inf - -inf.
  float m_run[HPL], l_run[HPL];
#pragma unroll
  for (int hh = 0; hh < HPL; ++hh) {
    m_run[hh] = -__FLT_MAX__;
    l_run[hh] = 0.f;
  }
  float acc[HG][EPL];
#pragma unroll
  for (int g = 0; g < HG; ++g)
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc[g][e] = 0.f;

  // One unit: scores, online softmax, PV.
  auto process = [&](const UnitRegs<NI, NC>& cur, int u) __attribute__((always_inline)) {
    const int base = t_begin + (u << UL);

    // ---- scores: partial q.k over this lane's EPL dims ----
    float part[NV];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      u32 kw[QW];
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        if constexpr (KV == KV_SAME) {
#pragma unroll
          for (int j = 0; j < 4; ++j) kw[n * QWC + j] = cur.k[i * NC + n][j];
        } else if constexpr (FOLD) {
          u32 o[8];
          k8_exact_f16<KV>(cur.k[i * NC + n], o);
#pragma unroll
          for (int j = 0; j < 8; ++j) kw[n * QWC + j] = o[j];
        } else {
          deq_pairs(cur.k[i * NC + n], cur.ksc[i], &kw[n * QWC]);
        }
      }
#pragma unroll
      for (int g = 0; g < HG; ++g) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < QW; ++j) {
          if constexpr (F32Q) s = __builtin_fmaf(as_f32(qv[g][j]), as_f32(kw[j]), s);
          else s = Pair<QT>::dot2(qv[g][j], kw[j], s);
        }
        part[g * NI + i] = FOLD ? s * cur.ksc[i] : s;  // load i's rows share one page
      }
    }
    transpose_reduce<LPR, NV>(part, c);

    // ---- online softmax (state shared by the wave, per head) ----
    float pr[NPL];
    float alpha[HPL];
#pragma unroll
    for (int hh = 0; hh < HPL; ++hh) {
      float mx = -INFINITY;
#pragma unroll
      for (int v = 0; v < VPH; ++v) {
        const int k = hh * VPH + v;
        const int j = c * NPL + k;
        const int i = j % NI;
        const bool valid = base + i * RPL + r < t_end;
        const float s = valid ? part[k] * p.scale_log2 : -INFINITY;
        pr[k] = s;
        mx = fmaxf(mx, s);
      }
      mx = within_quad<OpMax, LPH>(mx);
      mx = across_rows<OpMax, LPR>(mx);
      // Lazy max: m moves (and acc / l are rescaled) only when a unit's max
      // exceeds it by more than kDecLazy, so p = 2^(s - m) stays below
      // 2^kDecLazy -- exact in the fp32 sums and PV -- and most units skip
      // the rescale.
      const bool grow = mx > m_run[hh] + kDecLazy;
      const float m_new = grow ? mx : m_run[hh];
      alpha[hh] = grow ? fast_exp2(m_run[hh] - m_new) : 1.f;
      float ps = 0.f;
#pragma unroll
      for (int v = 0; v < VPH; ++v) {
        const int k = hh * VPH + v;
        pr[k] = fast_exp2(pr[k] - m_new);
        ps += pr[k];
      }
      l_run[hh] = l_run[hh] * alpha[hh] + ps;
      m_run[hh] = m_new;
    }

    // ---- broadcast p (per row) and alpha (per wave) through LDS ----
#pragma unroll
    for (int k = 0; k < NPL; ++k) s_p[w][r][c * NPL + k] = pr[k];
    if (r == 0) {
#pragma unroll
      for (int hh = 0; hh < HPL; ++hh) {
        const int j0 = c * NPL + hh * VPH;
        if (j0 % NI == 0) s_alpha[w][j0 / NI] = alpha[hh];
      }
    }
    wave_lds_fence();
    float pv[NV];
    float al[HG];
#pragma unroll
    for (int j = 0; j < NV; j += 4) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(&s_p[w][r][j]);
      pv[j] = t[0];
      pv[j + 1] = t[1];
      pv[j + 2] = t[2];
      pv[j + 3] = t[3];
    }
#pragma unroll
    for (int g = 0; g < HG; g += 4) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(&s_alpha[w][g]);
      al[g] = t[0];
      al[g + 1] = t[1];
      al[g + 2] = t[2];
      al[g + 3] = t[3];
    }
    wave_lds_fence();

    // ---- acc = acc * alpha + sum_i p_i * v_i (fp32) ----
    // al[] is the same for every lane of the wave (read back from LDS).
    bool rescale = false;
#pragma unroll
    for (int g = 0; g < HG; ++g) rescale |= al[g] != 1.f;
    if (rescale) {
#pragma unroll
      for (int g = 0; g < HG; ++g)
#pragma unroll
        for (int e = 0; e < EPL; ++e) acc[g][e] *= al[g];
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      float vf[EPL];
      u32 vw[QW];
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        if constexpr (KV == KV_SAME) {
#pragma unroll
          for (int j = 0; j < 4; ++j) vw[n * QWC + j] = cur.v[i * NC + n][j];
        } else {
          deq_pairs(cur.v[i * NC + n], cur.vsc[i], &vw[n * QWC]);
        }
      }
#pragma unroll
      for (int j = 0; j < QW; ++j) {
        if constexpr (F32Q) {
          vf[j] = as_f32(vw[j]);
        } else {
          vf[2 * j] = Pair<QT>::lo(vw[j]);
          vf[2 * j + 1] = Pair<QT>::hi(vw[j]);
        }
      }
#pragma unroll
      for (int g = 0; g < HG; ++g) {
        const float pg = pv[g * NI + i];
#pragma unroll
        for (int e = 0; e < EPL; ++e) acc[g][e] = __builtin_fmaf(pg, vf[e], acc[g][e]);
      }
    }
  };

  // Two register sets, unit u + NW loading while unit u is processed (the
  // loop is unrolled by two so that no copy moves one set into the other).
  UnitRegs<NI, NC> nxt;
  if constexpr (LANE) {
    if (!early && w < n_units) lookup(t_begin + (w << UL), t_end);
  }
  if (w < n_units) fetch(nxt, w, true);
  for (int u = w; u < n_units; u += NW) {
    UnitRegs<NI, NC> cur = nxt;
    if (u + NW < n_units) fetch(nxt, u + NW, false);
    if constexpr (LANE) {
      // Rows past t_end hold other tokens' data: their scores are masked,
      // and zero V rows keep p * v = 0 (the per-load form reads zeros there).
      // So do zero scales: a first unit can look its rows up before t_end is
      // known, in table columns that the sequence may not use, whose pages'
      // scales can be anything.
      if (t_begin + ((u + 1) << UL) > t_end) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const bool in = t_begin + (u << UL) + i * RPL + r < t_end;
          if constexpr (KV != KV_SAME && !BAL) cur.vsc[i] = in ? cur.vsc[i] : 0.f;
#pragma unroll
          for (int n = 0; n < NC; ++n)
#pragma unroll
            for (int j = 0; j < 4; ++j) cur.v[i * NC + n][j] = in ? cur.v[i * NC + n][j] : 0u;
        }
      }
    }
    process(cur, u);
  }

  // ---- merge rows of the wave (same m), then the waves of the workgroup ----
#pragma unroll
  for (int hh = 0; hh < HPL; ++hh) {
    float l = within_quad<OpAdd, LPH>(l_run[hh]);
    l_run[hh] = across_rows<OpAdd, LPR>(l);
  }
#pragma unroll
  for (int g = 0; g < HG; ++g)
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc[g][e] = across_rows<OpAdd, LPR>(acc[g][e]);
  if (r == 0) {
#pragma unroll
    for (int g = 0; g < HG; ++g)
#pragma unroll
      for (int e = 0; e < EPL; ++e) s_red[w][g][(c + LPR * (e / EPC)) * EPC + e % EPC] = acc[g][e];
#pragma unroll
    for (int hh = 0; hh < HPL; ++hh) {
      const int j0 = c * NPL + hh * VPH;
      if (j0 % NI == 0) {
        s_ml[w][j0 / NI][0] = m_run[hh];
        s_ml[w][j0 / NI][1] = l_run[hh];
      }
    }
  }
  __syncthreads();

  for (int idx = threadIdx.x; idx < HG * D; idx += NW * 64) {
    const int g = idx / D;
    const int d = idx % D;
    if (g >= nvalid) continue;
    float M = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) M = fmaxf(M, s_ml[ww][g][0]);
    float A = 0.f, L = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) {
        const float f = fast_exp2(s_ml[ww][g][0] - M);
        A = __builtin_fmaf(s_red[ww][g][d], f, A);
        L = __builtin_fmaf(s_ml[ww][g][1], f, L);
      }
    }
    const int h = head0 + g;
    if (BAL ? slot < 0 : S == 1) {
      store_elem<QT>(p.out, b * p.o_sb + h * p.o_sh + d, L > 0.f ? A / L : 0.f);
    } else if constexpr (BAL) {
      ws_store(const_cast<float*>(bal_acc(p, blockIdx.x, slot, g, D)) + d, A, true);
      if (d == 0) {
        float* ml = const_cast<float*>(bal_ml(p, blockIdx.x, slot, g));
        ws_store(ml, M, true);
        ws_store(ml + 1, L, true);
      }
    } else {
      const int64_t row = ((int64_t)b * p.H + h) * S + split;
      const bool coh = p.counters != nullptr;
      ws_store(p.ws_acc + row * D + d, A, coh);
      if (d == 0) {
        ws_store(p.ws_ml + row * 2 + 0, M, coh);
        ws_store(p.ws_ml + row * 2 + 1, L, coh);
      }
    }
  }
  if constexpr (BAL) {
    __shared__ float s_f[kBalRows * 64], s_mm[kBalRows * 2];
    if (slot >= 0)
      bal_merge<QT, D, NW * 64>(p, item, w_first, n_parts, nvalid,
                                [&](int j) { return (int64_t)b * p.o_sb + (int64_t)(head0 + j) * p.o_sh; }, s_f, s_mm);
  } else if (S > 1 && p.counters) {
    merge_in_launch<QT, D>(p, S, b * gridDim.y + y, nvalid, [&](int j, int64_t& bh, int64_t& o) {
      const int h = head0 + j;
      bh = (int64_t)b * p.H + h;
      o = (int64_t)b * p.o_sb + (int64_t)h * p.o_sh;
    });
  }
  };  // segment

  if constexpr (BAL) {
    constexpr int WB = Gm::kUnitLog2 + (NW == 8 ? 3 : 2);  // a block: one unit per wave
    bal_run<NW * 64, WB>(p, [&](const DecodeParams& q, int b, int y, int t_begin, int t_end, int slot, int item,
                                int w_first, int n) __attribute__((always_inline)) {
                                  segment(q, b, y, 0, 1, t_begin, t_end, slot, item, w_first, n);
                                });
  } else {
    int b, y, split;
    partition_item(p, b, y, split);
    segment(p, b, y, split, gridDim.x, 0, 0, 0, 0, 0, 0);
  }
}

// ---------------------------------------------------------------------------
// MFMA decode for large GQA groups (group >= 8, e.g. MQA 32/1): one workgroup
// per (partition, KV head, up to 32 of its query heads, sequence).  With G
// query heads per KV head every K/V byte feeds 2G FLOPs, more than the VALU
// sustains at HBM speed for G >= 8, so both products run on the matrix core:
//   S^T = K Q^T   v_mfma_f32_32x32x16: A = 32 keys x 16 dims straight from
//                 each lane's own 16-byte K loads (the head dims are permuted
//                 identically in K and Q so those loads stay contiguous),
//                 B = Q^T of the 32 heads (registers, loaded once);
//   O^T += V^T P^T  A = V^T through the wave's LDS tile (ds_read_b64_tr_b16),
//                 B = P^T straight from the S^T accumulator.
// Each wave streams its own 32-key blocks (wave-private LDS, no workgroup
// barrier in the loop) with its own online softmax; the waves merge at the
// end, and partitions go through the same log-sum-exp merge as the VALU
// kernel.  P is rounded to the K/V type for PV (bf16: hi + lo parts).
// ---------------------------------------------------------------------------
// NW = 4 or 8 waves per workgroup: the host takes 8 when the grid has fewer
// than two workgroups per CU, so each CU still streams 8 blocks at a time.
template <typename QT, int KV, int D, int NW, bool BAL = false>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
void paged_decode_mfma_kernel(const DecodeParams p) {
  constexpr int KS = D / 16;     // MFMA k-steps
  constexpr int DB = D / 32;     // 32-dim blocks of O^T
  constexpr int K_RS = D + 8;    // LDS row strides (elements) of the K and V
  constexpr int V_RS = D + 32;   // tiles, spreading reads over the banks
  constexpr bool SPLIT_P = std::is_same<QT, BF16>::value;
  constexpr int EB = KV == KV_SAME ? 2 : 1;        // bytes per stored element
  // Row-coalesced loads: CPR lanes cover one stored row with 16-byte chunks
  // (EPC elements each); one load instruction covers RPL rows, so a 32-key
  // block takes NLD loads per lane for K and as many for V.
  constexpr int EPC = 16 / EB;
  constexpr int CPR = D / EPC;
  constexpr int RPL = 64 / CPR;
  constexpr int NLD = 32 / RPL;
  static_assert(CPR * EPC == D && NLD * RPL == 32, "unsupported head_dim / element size");

  // K and V tiles during the loop; per-wave O / m / l for the merge after it.
  constexpr int kTileBytes = NW * 32 * (K_RS + V_RS) * 2;
  constexpr int OS = D + 4;  // O's row stride (floats): 32 rows' 16-byte pieces hit distinct banks
  constexpr int kMergeBytes = (NW * 32 * OS + NW * 32 * 2) * 4;
  __shared__ __attribute__((aligned(16))) uint8_t smem[kTileBytes > kMergeBytes ? kTileBytes : kMergeBytes];

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 31;  // key row (A operand) / (head, token) column (B, S^T)
  const int g = lane >> 5;   // k-group: head dims 16ks + 8g .. +7 of k-step ks

  // One partition, or segment (see paged_decode_kernel), to "// segment".
  auto segment = [&](const DecodeParams& p, const int b, const int y, const int split, const int S, const int seg_begin, const int seg_end,
                     const int slot, const int item, const int w_first, const int n_parts)
      __attribute__((always_inline)) {
  const int sub = y % p.hg_per_kv;
  const int kvh = y / p.hg_per_kv;
  // The workgroup's 32 columns are rows r = sub * 32 + c of this KV head's
  // group * T (query head, token) pairs: head kvh * group + r % group, token
  // r / group (T = 1: the heads of the group).
  const int row_base = sub * 32;
  const int nvalid = min(32, p.group * p.T - row_base);

  // Page ids of this wave's first 32-key block, read together with seq_len
  // when `early` (first_page_ids).
  const int32_t* ptrow = p.pt + (int64_t)b * p.pt_sb;
  const bool early = !BAL && (split == 0 || p.pps_fixed > 0);
  int first_pid[NLD];
  int seq_len, t_begin, t_end;
  if constexpr (BAL) {
    seq_len = max(0, min(uniform_load(p.lens, b), p.max_pages << p.log2P));
    t_begin = seg_begin;
    t_end = seg_end;
  } else {
    seq_len = first_page_ids<NLD, RPL>(first_pid, ptrow, p, split, w << 5, b, early);
    seq_len = max(0, min(seq_len, p.max_pages << p.log2P));
    const int np = (seq_len + p.P - 1) >> p.log2P;
    const int pps = p.pps_fixed > 0 ? p.pps_fixed : (np + S - 1) / S;
    const int pb = split * pps;
    const int pe = split == S - 1 ? np : min(np, pb + pps);
    t_begin = pb << p.log2P;
    t_end = min(seq_len, pe << p.log2P);
  }
  const int n_blocks = t_end > t_begin ? (t_end - t_begin + 31) >> 5 : 0;
  // This lane's column: (query head, token) and the end of its visible keys.
  const int my_r = row_base + min(li, nvalid - 1);
  const int my_t = my_r / p.group;
  const int my_h = kvh * p.group + (my_r - my_t * p.group);
  const int my_end = min(t_end, seq_len - p.T + 1 + my_t);

  // Q^T: lane (column li, k-group g), k-step ks = head dims 16ks + 8g + 0..7.
  u32x4 qf[KS];
  {
    const uint8_t* qp = p.q + 2 * ((int64_t)b * p.q_sb + (int64_t)my_t * p.q_st + (int64_t)my_h * p.q_sh + 8 * g);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const u32x4*>(qp + 32 * ks);
  }

  const int lrow = lane / CPR;  // this lane's row inside each load
  const int lcol = lane % CPR;  // and its 16-byte chunk
  // Raw K/V chunks of a 32-key block: load i covers rows RPL*i .. RPL*i +
  // RPL - 1, which lie in one page (page_size >= RPL), so its page id and
  // (8-bit caches) scales are wave-uniform.  Its address is that page's
  // base (scalar unit, in a buffer descriptor) plus this lane's
  // loop-invariant offset; the descriptor's range ends with the partition's
  // last row, so rows past t_end read as zeros (their scores are masked, and
  // zero bytes are zero in every cache type).
  const uint8_t* const kh = p.k + (int64_t)EB * kvh * p.k_sh;  // this KV head's slice of page 0
  const uint8_t* const vh = p.v + (int64_t)EB * kvh * p.v_sh;
  const uint32_t kpage = (uint32_t)(EB * p.k_sp), vpage = (uint32_t)(EB * p.v_sp);
  const uint32_t krow = (uint32_t)(EB * p.k_ss), vrow = (uint32_t)(EB * p.v_ss);
  const uint32_t lane_k = lrow * krow + 16 * lcol;
  const uint32_t lane_v = lrow * vrow + 16 * lcol;
  struct Raw {
    u32x4 k[NLD], v[NLD];
    float ksc[NLD], vsc[NLD];
  };
  // first: blk is this wave's first block (first_pid holds its page ids).
  auto fetch = [&](Raw& R, int blk, bool first) {
    const int kb = t_begin + (blk << 5);
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int rs = kb + i * RPL;
      const int nrow = min(t_end - rs, RPL);  // rows of this load in the partition
      // read without a branch (at most the table's last entry); a load wholly
      // past t_end reads nothing (range 0), 8-bit caches the page of a row
      // before it (see paged_decode_kernel)
      int phys;
      if constexpr (KV == KV_SAME)
        phys = first && early ? first_pid[i] : uniform_load(ptrow, min(rs >> p.log2P, p.max_pages - 1));
      else
        phys = first && early ? (nrow > 0 ? first_pid[i] : first_pid[0])
                              : uniform_load(ptrow, min(rs, t_end - 1) >> p.log2P);
      phys = __builtin_amdgcn_readfirstlane(min(max(phys, 0), p.num_pages - 1));
      const uint32_t slot0 = (uint32_t)(rs & (p.P - 1));
      const int nk = nrow > 0 ? (int)((uint32_t)(nrow - 1) * krow + EB * D) : 0;
      const int nv = nrow > 0 ? (int)((uint32_t)(nrow - 1) * vrow + EB * D) : 0;
      R.k[i] = kv_buffer_load(kh + (uint64_t)(uint32_t)phys * kpage + slot0 * krow, nk, lane_k);
      R.v[i] = kv_buffer_load(vh + (uint64_t)(uint32_t)phys * vpage + slot0 * vrow, nv, lane_v);
      if constexpr (KV != KV_SAME) {
        R.ksc[i] = uniform_load(p.ks, (int64_t)phys * p.sc_sp + (int64_t)kvh * p.sc_sh);
        R.vsc[i] = uniform_load(p.vs, (int64_t)phys * p.sc_sp + (int64_t)kvh * p.sc_sh);
      }
    }
  };
  // FOLD (8-bit cache, fp16 queries): exact 8-bit K and k_scale on the
  // scores (k8_exact_f16).  int8 V as x * fp16(v_scale), one packed fp16
  // multiply per pair (FOLD_V): within one fp16 ulp of round_to_fp16(
  // float(x) * v_scale) (the scale's own rounding to fp16 is the second
  // rounding; a scale below fp16's normal range, 6.1e-5, can be off by up to
  // 3e-8, i.e. a V error below 4e-6), inside the dequantise-then-attend
  // tolerance.  fp8 V keeps the fp32 dequantise, which measured faster there.
  constexpr bool FOLD = KV != KV_SAME && std::is_same<QT, F16>::value;
  constexpr bool FOLD_V = FOLD && KV == KV_I8;
  // Store one raw chunk as QT elements at dst (EPC of them): a copy for
  // fp16/bf16 caches, round_to_QT(float(x) * scale) for 8-bit ones, or
  // (put_exact, FOLD K) the exact 8-bit values.
  auto put_exact = [&](uint16_t* dst, const u32x4& raw) {
    u32 o[8];
    k8_exact_f16<KV>(raw, o);
    *reinterpret_cast<u32x4*>(dst) = u32x4{o[0], o[1], o[2], o[3]};
    *reinterpret_cast<u32x4*>(dst + 8) = u32x4{o[4], o[5], o[6], o[7]};
  };
  auto put_scaled = [&](uint16_t* dst, const u32x4& raw, float sc) {
    u32 o[8];
    k8_exact_f16<KV>(raw, o);
    const f16x2 s2 = {(f16)sc, (f16)sc};
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = __builtin_bit_cast(u32, __builtin_bit_cast(f16x2, o[j]) * s2);
    *reinterpret_cast<u32x4*>(dst) = u32x4{o[0], o[1], o[2], o[3]};
    *reinterpret_cast<u32x4*>(dst + 8) = u32x4{o[4], o[5], o[6], o[7]};
  };
  auto put = [&](uint16_t* dst, const u32x4& raw, float sc) {
    if constexpr (KV == KV_SAME) {
      *reinterpret_cast<u32x4*>(dst) = raw;
    } else {
      const float nb = -128.0f * sc;
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) {
        u32x4 o;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          float f[4];
          if constexpr (KV == KV_I8) {
            i8x4_biased(raw[2 * h2 + j], f);
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = __builtin_fmaf(f[e], sc, nb);
          } else {
            fp8x4(raw[2 * h2 + j], f);
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = f[e] * sc;
          }
          o[2 * j] = Pair<QT>::pack(f[0], f[1]);
          o[2 * j + 1] = Pair<QT>::pack(f[2], f[3]);
        }
        *reinterpret_cast<u32x4*>(dst + 8 * h2) = o;
      }
    }
  };

  uint16_t* const Kt = reinterpret_cast<uint16_t*>(smem) + w * 32 * (K_RS + V_RS);
  uint16_t* const Vt = Kt + 32 * K_RS;
  const int tr_c = (lane & 15) >> 2;
  const int tr_j = lane & 3;
  const int tr_G = lane >> 4;
  const int tr_row = 4 * (tr_G >> 1) + tr_c;
  const int tr_col = 16 * (tr_G & 1) + 4 * tr_j;

  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
  float m_run = -INFINITY;  // log2 units
  float l_run = 0.f;
  const float c = p.scale_log2;

  // One 32-key block from R; refills R with block nxt once R is consumed.
  auto compute = [&](Raw& R, int blk, int nxt) {
    // K(blk) and V(blk) into this wave's LDS tiles (row = key, columns =
    // head dims), then R is free for the next block's loads.
    float ck[NLD];  // FOLD: score factor (softmax scale times k_scale) per load
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int row = i * RPL + lrow;
      if constexpr (FOLD) {
        ck[i] = c * R.ksc[i];
        put_exact(&Kt[row * K_RS + lcol * EPC], R.k[i]);
      } else {
        put(&Kt[row * K_RS + lcol * EPC], R.k[i], R.ksc[i]);
      }
      if constexpr (FOLD_V) {
        put_scaled(&Vt[row * V_RS + lcol * EPC], R.v[i], R.vsc[i]);
      } else {
        put(&Vt[row * V_RS + lcol * EPC], R.v[i], R.vsc[i]);
      }
    }
    if (nxt < n_blocks) fetch(R, nxt, false);
    wave_lds_fence();
    // S^T = K Q^T for the 32 keys of this block: A = K rows li, dims 16ks + 8g.
    f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const u32x4 a = *reinterpret_cast<const u32x4*>(&Kt[li * K_RS + 16 * ks + 8 * g]);
      s = Mfma<QT>::mma(a, qf[ks], s);
    }

    // Online softmax for column li over keys kb + (r&3) + 4g + 8(r>>2).
    const int kb = t_begin + (blk << 5);
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = kb + (r & 3) + 4 * g + 8 * (r >> 2);
      // key row 8 (r >> 2) + (r & 3) + 4g of the block: load (r >> 2) * 8 / RPL
      const float cr = FOLD ? ck[(r >> 2) * 8 / RPL] : c;
      const float x = key < my_end ? s[r] * cr : -INFINITY;
      s[r] = x;
      mx = fmaxf(mx, x);
    }
    mx = xor32<OpMax>(mx);
    if (__any(mx > m_run + kDecLazy)) {
      const bool grow = mx > m_run + kDecLazy;
      const float alpha = grow ? fast_exp2(m_run - mx) : 1.f;
      m_run = grow ? mx : m_run;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
    }
    // A column that has seen no visible key yet (only possible for T > 1)
    // keeps m = -inf; its scores are -inf too, and exp2(-inf - 0) = 0.
    const float m_use = m_run == -INFINITY ? 0.f : m_run;
    u32x4 pf[2], pl[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        const float x0 = fast_exp2(s[8 * t + 2 * e2] - m_use);
        const float x1 = fast_exp2(s[8 * t + 2 * e2 + 1] - m_use);
        l_run += x0 + x1;
        const u32 hp = Pair<QT>::pack(x0, x1);
        pf[t][e2] = hp;
        if constexpr (SPLIT_P) pl[t][e2] = Pair<QT>::pack(x0 - Pair<QT>::lo(hp), x1 - Pair<QT>::hi(hp));
      }
    wave_lds_fence();
    // O^T += V^T P^T (k-step t covers keys 16t..16t+15 of the block).
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int vrow = 16 * t + tr_row;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const uint16_t* vp = &Vt[vrow * V_RS + 32 * db + tr_col];
        const u32x2 lo = lds_read_tr16(vp);
        const u32x2 hi2 = lds_read_tr16(vp + 8 * V_RS);
        const u32x4 a = {lo[0], lo[1], hi2[0], hi2[1]};
        acc[db] = Mfma<QT>::mma(a, pf[t], acc[db]);
        if constexpr (SPLIT_P) acc[db] = Mfma<QT>::mma(a, pl[t], acc[db]);
      }
    }
    wave_lds_fence();
  };
  Raw R;
  if (w < n_blocks) fetch(R, w, true);
  for (int blk = w; blk < n_blocks; blk += NW) compute(R, blk, blk + NW);

  // ---- merge the waves: O = sum_w acc_w 2^(m_w - M) / sum_w l_w 2^(m_w - M) ----
  __syncthreads();  // every wave is done with its V tile (smem is reused)
  float* so = reinterpret_cast<float*>(smem);   // [NW][32 columns][OS]
  float* sml = so + NW * 32 * OS;               // [NW][32 columns][2]
  const float l_tot = xor32<OpAdd>(l_run);
  // Four dims of a column per write, the valid columns only (one dword per
  // write and a row stride of D floats put 32 lanes in one bank, 7 us of a
  // launch's end with 8 waves).
  if (li < nvalid) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        *reinterpret_cast<f32x4*>(&so[(w * 32 + li) * OS + 32 * db + 4 * g + 8 * r4]) =
            f32x4{acc[db][4 * r4], acc[db][4 * r4 + 1], acc[db][4 * r4 + 2], acc[db][4 * r4 + 3]};
  }
  if (g == 0) {
    sml[(w * 32 + li) * 2 + 0] = m_run;
    sml[(w * 32 + li) * 2 + 1] = l_tot;
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < nvalid * D; idx += NW * 64) {
    const int hh = idx / D;
    const int d = idx - hh * D;
    float M = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) M = fmaxf(M, sml[(ww * 32 + hh) * 2]);
    float A = 0.f, L = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) {
        const float f = fast_exp2(sml[(ww * 32 + hh) * 2] - M);
        A = __builtin_fmaf(so[(ww * 32 + hh) * OS + d], f, A);
        L = __builtin_fmaf(sml[(ww * 32 + hh) * 2 + 1], f, L);
      }
    }
    const int rr = row_base + hh;
    const int tt = rr / p.group;
    const int h = kvh * p.group + (rr - tt * p.group);
    if (BAL ? slot < 0 : S == 1) {
      uint16_t* op = reinterpret_cast<uint16_t*>(p.out) + (b * p.o_sb + tt * p.o_st + h * p.o_sh + d);
      *op = Pair<QT>::from_float(L > 0.f ? A / L : 0.f);
    } else if constexpr (BAL) {
      ws_store(const_cast<float*>(bal_acc(p, blockIdx.x, slot, hh, D)) + d, A, true);
      if (d == 0) {
        float* ml = const_cast<float*>(bal_ml(p, blockIdx.x, slot, hh));
        ws_store(ml, M, true);
        ws_store(ml + 1, L, true);
      }
    } else {
      const int64_t row = (((int64_t)b * p.T + tt) * p.H + h) * S + split;
      const bool coh = p.counters != nullptr;
      ws_store(p.ws_acc + row * D + d, A, coh);
      if (d == 0) {
        ws_store(p.ws_ml + row * 2 + 0, M, coh);
        ws_store(p.ws_ml + row * 2 + 1, L, coh);
      }
    }
  }
  if constexpr (BAL) {
    if (slot >= 0) {  // the tiles are free: the merge's barriers come first
      float* const s_f = sml + NW * 32 * 2;
      static_assert((NW * 32 * OS + NW * 32 * 2 + kBalRows * 66) * 4 <= (int)sizeof(smem), "merge weights");
      bal_merge<QT, D, NW * 64>(p, item, w_first, n_parts, nvalid, [&](int j) {
        const int rr = row_base + j;
        const int tt = rr / p.group;
        const int h = kvh * p.group + (rr - tt * p.group);
        return (int64_t)b * p.o_sb + (int64_t)tt * p.o_st + (int64_t)h * p.o_sh;
      }, s_f, s_f + kBalRows * 64);
    }
  } else if (S > 1 && p.counters) {
    merge_in_launch<QT, D>(p, S, b * gridDim.y + y, nvalid, [&](int j, int64_t& bh, int64_t& o) {
      const int rr = row_base + j;
      const int tt = rr / p.group;
      const int h = kvh * p.group + (rr - tt * p.group);
      bh = ((int64_t)b * p.T + tt) * p.H + h;
      o = (int64_t)b * p.o_sb + (int64_t)tt * p.o_st + (int64_t)h * p.o_sh;
    });
  }
  };  // segment

  if constexpr (BAL) {
    constexpr int WB = 5 + (NW == 8 ? 3 : 2);  // a block: 32 keys per wave
    bal_run<NW * 64, WB>(p, [&](const DecodeParams& q, int b, int y, int t_begin, int t_end, int slot, int item,
                                int w_first, int n) __attribute__((always_inline)) {
                                  segment(q, b, y, 0, 1, t_begin, t_end, slot, item, w_first, n);
                                });
  } else {
    int b, y, split;
    partition_item(p, b, y, split);
    segment(p, b, y, split, gridDim.x, 0, 0, 0, 0, 0, 0);
  }
}

}  // namespace fat
