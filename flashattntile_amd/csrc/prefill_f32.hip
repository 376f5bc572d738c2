// prefill_f32.hip -- packed fp32 prefill on the fp32 matrix instructions
// (v_mfma_f32_32x32x2_f32), head_dim 32, 64 and 128.
//
// Semantics are those of the other prefill kernels (flashattn_tile/kernels/
// prefill.py:35-138; the reference runs fp32 through its fp32 torch path,
// kernels/prefill.py:286-290): scores, softmax and PV in fp32, P not rounded.
//
// What bounds it: the fp32 matrix rate, 157 TFLOP/s at 2.4 GHz, twice what
// scalar fp32 FMAs reach.  A 32x32x2 MFMA takes 64 cycles and one dword of
// each operand per lane, so neither LDS nor the loads are near their limits;
// what has to be kept short is a query block's chain of key tiles and the
// time a SIMD spends in the softmax.
//
// Design: one workgroup of four waves per block of 32 query rows and query
// head; wave w takes key tiles w, w + 4, ... (32 keys each) and the four
// partial results are merged by log-sum-exp at the end.  Splitting the keys
// instead of giving each wave rows of its own makes the longest chain a
// quarter as long and the grid four times as large, which is what ragged
// packs of a few sequences need (one block of 128 rows per workgroup would
// hold a SIMD for 38 tiles at 1212 keys, longer than the whole launch takes
// now).
//   * K tiles go straight into wave-private LDS (buffer_load ... lds, no
//     registers, no workgroup barrier in the loop), K(t + 4) during softmax
//     and PV of tile t.  Chunk c of row r sits in slot c ^ r (of 16 bytes),
//     so the operand reads hit distinct banks without padding;
//   * S^T = K Q^T: a lane reads four consecutive dims of its key row at once
//     and Q's registers follow the same order of dims;
//   * O^T += V^T P^T: accumulator register r of S^T holds keys k and k + 4 of
//     the two lane halves, which is one k-step's P^T operand as it stands;
//     block db of O^T holds dims DB m + db, so a lane's V^T operands of all
//     blocks are consecutive floats: one row-coalesced load from memory into
//     registers, no LDS;
//   * LDS and registers leave room for two workgroups per CU, so one wave of
//     a SIMD runs its softmax, waits and merge under the other's MFMAs.
// Measured against the VALU kernel of prefill_generic.hip (32/8 heads, D128,
// causal): one sequence of 4096 2.55 -> 1.15 ms (119 TFLOP/s; the matrix pipe
// is busy 82 % of its cycles, at 2.2 GHz), a pack of 375 + 775 + 1212 391 ->
// 206 us, where the blocks' start-up and the merge weigh more.
#include "prefill_common.h"

namespace fat {

typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kF32BM = 32;  // query rows per workgroup
constexpr int kF32BN = 32;  // keys per tile
constexpr float kF32Lazy = 8.0f;  // lazy-rescale bound (log2 units)

template <int D, bool CAUSAL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 128 ? 2 : 3, D == 128 ? 2 : 3)))
void prefill_f32_kernel(const PrefillParams p) {
  constexpr int NW = 4;
  constexpr int DB = D / 32;           // 32-row blocks of O^T
  constexpr int CPR = D / 4;           // 16-byte chunks per row
  constexpr int RB = 4 * D;            // row bytes
  constexpr int TILE = kF32BN * RB;    // bytes of a K tile
  constexpr int NL = TILE / 1024;      // loads per tile
  constexpr int RPLD = 64 / CPR;       // rows per load
  constexpr int RDIV = CPR >= 16 ? 1 : 16 / CPR;  // rows that share a swizzle (they differ in banks anyway)
  // A score is two independent sums, so that rounding grows no faster than
  // in the VALU kernel.  Distance of the output from 64 bits (777 causal
  // keys, D128): one sum 6.6e-7, two 4.5e-7, four 3.7e-7 (with spills), the
  // VALU kernel 5.9e-7.
  constexpr int SC = 2;
  static_assert(kF32BM == kF32BN, "a wave's partial output takes the place of its K tile");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[NW * TILE];
  __shared__ float s_ml[NW][kF32BM][2];

  const int per = p.B * p.H;
  const int jb = blockIdx.x / per;
  const int rem = blockIdx.x - jb * per;
  const int b = rem / p.H;
  const int j = rem - b * p.H;
  const int kvh = j % p.Hkv;  // heads that share a KV head land on one XCD
  const int h = kvh * p.group + j / p.Hkv;

  const int q_start = p.cu_q[b];
  const int q_len = p.cu_q[b + 1] - q_start;
  const int k_start = p.cu_k[b];
  const int kv_len = p.cu_k[b + 1] - k_start;
  // Blocks are counted from the sequence's last row, longest causal chain
  // first; rows below 0 of its last block compute as row 0 and aren't stored.
  if (jb * kF32BM >= q_len) return;  // uniform over the workgroup
  const int r_end = q_len - jb * kF32BM;
  const int row0 = r_end - kF32BM;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;
  const int li = lane & 31;
  const int shift = kv_len - q_len;
  const float c = p.scale_log2;

  int hi = kv_len;
  if (CAUSAL) hi = min(kv_len, r_end + shift);
  const int n_tiles = hi > 0 ? (hi + kF32BN - 1) / kF32BN : 0;

  // The sequence's rows of this KV head; rows past kv_len - 1 read as zeros
  // (their scores are masked, and zero V rows keep p * v = 0).
  const int kst = (int)(4 * p.k_st), vst = (int)(4 * p.v_st);
  const uint64_t kseq = reinterpret_cast<uint64_t>(p.k + 4 * ((int64_t)k_start * p.k_st + (int64_t)kvh * p.k_sh));
  const uint8_t* const vseq = p.v + 4 * ((int64_t)k_start * p.v_st + (int64_t)kvh * p.v_sh);
  auto range = [&](int st) { return (int)min((int64_t)max(kv_len - 1, 0) * st + RB, (int64_t)0x7fffffff); };
  const i32x4 kdesc = {__builtin_amdgcn_readfirstlane((int)(uint32_t)kseq),
                       __builtin_amdgcn_readfirstlane((int)((uint32_t)(kseq >> 32) & 0xffffu)),
                       __builtin_amdgcn_readfirstlane(range(kst)), kBufFlags};
  const __amdgpu_buffer_rsrc_t vdesc = __builtin_amdgcn_make_buffer_rsrc((void*)vseq, (short)0, range(vst), kBufFlags);
  uint8_t* const Kt = lds + w * TILE;
  const int kt_addr = (int)(uintptr_t)(lds_void*)Kt;

  // Load i of a tile fills slots 64 i + lane: row RPLD i + lane / CPR, slot
  // lane % CPR, which holds chunk slot ^ ((row / RDIV) % CPR).
  const int lrow = lane / CPR;
  const int lchunk = 16 * ((lane % CPR) ^ (lrow / RDIV));
  auto issue_k = [&](int t) __attribute__((always_inline)) {
    int lc = lchunk;
    __asm__ volatile("" : "+v"(lc));  // per-load offsets are made here, not kept over the loop
    const int row_off = lrow * kst + t * kF32BN * kst;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int xi = 16 * (((RPLD * i) / RDIV) & (CPR - 1));
      buffer_load_lds16(kdesc, (lc ^ xi) + (row_off + RPLD * i * kst), kt_addr + 1024 * i);
    }
  };

  // Q^T, the B operand: dims 8 jj + 4 g + e of row li.
  float qf[D / 2];
  {
    const int qr = max(row0 + li, 0);
    const float* qp = reinterpret_cast<const float*>(p.q) + (int64_t)(q_start + qr) * p.q_st + (int64_t)h * p.q_sh + 4 * g;
#pragma unroll
    for (int jj = 0; jj < D / 8; ++jj) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(qp + 8 * jj);
#pragma unroll
      for (int e = 0; e < 4; ++e) qf[4 * jj + e] = x[e];
    }
  }

  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  const int lim = CAUSAL ? min(kv_len - 1, max(row0 + li, 0) + shift) : kv_len - 1;  // last visible key
  const int lim0 = CAUSAL ? min(kv_len - 1, max(row0, 0) + shift) : kv_len - 1;      // of the block's first row
  const int kread = li * RB;
  const int kswz = 16 * (g ^ ((li / RDIV) & (CPR - 1)));
  const int vlane = 4 * g * vst + 4 * DB * li;

  // All LDS reads so far have returned: their tile may be overwritten.
  auto reads_done = [&]() __attribute__((always_inline)) {
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };

  // The wave of SIMD w starts at tile (w + block) % 4: where the tiles don't
  // divide by four, the odd ones go to another SIMD in the next block.
  const int t0 = (w + jb + rem) & (NW - 1);
  if (t0 < n_tiles) issue_k(t0);
  // Q's registers are complete here: the compiler, which doesn't count the
  // tile loads, would otherwise wait for it inside the loop, and with it for
  // the loads behind it.
#pragma unroll
  for (int i = 0; i < D / 2; ++i) __asm__ volatile("" : "+v"(qf[i]));
  for (int t = t0; t < n_tiles; t += NW) {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): K(t) is in LDS
    __asm__ volatile("" ::: "memory");   // no LDS read of it moves above the wait
    int ks = kswz, vl = vlane;
    __asm__ volatile("" : "+v"(ks), "+v"(vl));  // as for lc
    f32x16 sc[SC];
#pragma unroll
    for (int jj = 0; jj < D / 8; ++jj) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(Kt + kread + (ks ^ (32 * jj)));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f32x16 prev = jj == 0 && e < SC ? f32x16{} : sc[e % SC];
        sc[e % SC] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], qf[4 * jj + e], prev, 0, 0, 0);
      }
    }
    // Two operand reads ahead of their four MFMAs each.
    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
    for (int jj = 0; jj < D / 8; ++jj) {
      __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
      if (jj + 2 < D / 8) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = (sc[0][r] + sc[1][r]) * c;
    // V(t)'s rows take the registers that the partial scores leave (the
    // scheduler would load them earlier, and spill), then the next K tile.
    __builtin_amdgcn_sched_barrier(0);
    u32x4 vr[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int off = vl + (t * kF32BN + (r & 3) + 8 * (r >> 2)) * vst;
      if constexpr (DB == 4) {
        vr[r] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(vdesc, off, 0, 0));
      } else if constexpr (DB == 2) {
        const u32x2 x = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(vdesc, off, 0, 0));
        vr[r][0] = x[0];
        vr[r][1] = x[1];
      } else {
        vr[r][0] = __builtin_amdgcn_raw_buffer_load_b32(vdesc, off, 0, 0);
      }
    }
    reads_done();
    if (t + NW < n_tiles) issue_k(t + NW);

    // Online softmax of query li over keys n0 + (r & 3) + 8 (r >> 2) + 4 g.
    const int n0 = t * kF32BN;
    float mx = -INFINITY;
    if (n0 + kF32BN - 1 > lim0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = n0 + (r & 3) + 8 * (r >> 2) + 4 * g <= lim ? s[r] : -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = xor32<OpMax>(mx);
    // Lazy max: m moves when some row's max exceeds it by more than kF32Lazy,
    // so p stays below 2^kF32Lazy (exact in the fp32 sums and PV).
    if (__any(mx > m_run + kF32Lazy)) {
      const bool grow = mx > m_run + kF32Lazy;
      const float alpha = grow ? fast_exp2(m_run - mx) : 1.f;
      m_run = grow ? mx : m_run;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
    }
    // A row with no visible key yet keeps m = -inf; its scores are -inf too.
    const float m_use = m_run == -INFINITY ? 0.f : m_run;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r] - m_use);
      l_run += s[r];
    }

#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int db = 0; db < DB; ++db)
        acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(as_f32(vr[r][db]), s[r], acc[db], 0, 0, 0);
  }

  // Partial (O, m, l) of each wave into its own K tile (same slots), then
  // the merge.
  l_run = xor32<OpAdd>(l_run);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = (r & 3) + 8 * (r >> 2) + 4 * g;
    const int at = li * RB + 16 * ((DB * m / 4) ^ ((li / RDIV) & (CPR - 1))) + 4 * (DB * m % 4);
#pragma unroll
    for (int db = 0; db < DB; ++db) *reinterpret_cast<float*>(Kt + at + 4 * db) = acc[db][r];
  }
  if (g == 0) {
    s_ml[w][li][0] = m_run;
    s_ml[w][li][1] = l_run;
  }
  __syncthreads();
  const bool o16 = ((reinterpret_cast<uintptr_t>(p.out) | (uintptr_t)(4 * p.o_st) | (uintptr_t)(4 * p.o_sh)) & 15) == 0;
  for (int idx = tid; idx < kF32BM * CPR; idx += 256) {
    const int r = idx / CPR;
    const int ch = idx - r * CPR;
    if ((unsigned)(row0 + r) >= (unsigned)q_len) continue;
    float M = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) M = fmaxf(M, s_ml[ww][r][0]);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    if (M != -INFINITY) {
      float L = 0.f;
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) {
        const float f = fast_exp2(s_ml[ww][r][0] - M);  // 0 for a wave without a visible key
        const f32x4 x = *reinterpret_cast<const f32x4*>(lds + ww * TILE + r * RB + 16 * (ch ^ ((r / RDIV) & (CPR - 1))));
        L = __builtin_fmaf(s_ml[ww][r][1], f, L);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = __builtin_fmaf(x[e], f, o[e]);
      }
      const float inv = L > 0.f ? 1.f / L : 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] *= inv;
    }
    float* dst = reinterpret_cast<float*>(p.out) + (int64_t)(q_start + row0 + r) * p.o_st + (int64_t)h * p.o_sh + 4 * ch;
    if (o16) {
      *reinterpret_cast<f32x4*>(dst) = o;
    } else {
      *reinterpret_cast<f32x2*>(dst) = f32x2{o[0], o[1]};
      *reinterpret_cast<f32x2*>(dst + 2) = f32x2{o[2], o[3]};
    }
  }
}

}  // namespace fat

namespace fat_host {

template <int D>
static void launch_f32_d(const fat::PrefillParams& prm, bool causal, dim3 grid, hipStream_t stream) {
  if (causal) hipLaunchKernelGGL((fat::prefill_f32_kernel<D, true>), grid, dim3(256), 0, stream, prm);
  else hipLaunchKernelGGL((fat::prefill_f32_kernel<D, false>), grid, dim3(256), 0, stream, prm);
}

int launch_prefill_f32(const fat::PrefillParams& prm, int D, bool causal, dim3 grid, hipStream_t stream) {
  switch (D) {
    case 128: launch_f32_d<128>(prm, causal, grid, stream); break;
    case 64: launch_f32_d<64>(prm, causal, grid, stream); break;
    case 32: launch_f32_d<32>(prm, causal, grid, stream); break;
    default:
      set_error("prefill: the fp32 matrix kernel takes head_dim 32, 64 and 128, got %d", D);
      return FAT_E_UNSUPPORTED;
  }
  return launch_status("prefill_f32_kernel");
}

}  // namespace fat_host
