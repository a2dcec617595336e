// The row sums that a backward needs in front of its two launches, as a launch of its own: with AE_BWD_KIND 0 where the dq
// launch comes last (ae_bwd_dq.hip), for the other kinds always.  Needs AE_DV, AE_BWD_KIND, AE_BWD_NRS.

#ifndef AE_BWD_DELTA_H
#define AE_BWD_DELTA_H

// Work buffer fp32 [2,B,Hq,Sq]: plane 0 = rowsum(do * o) (softmax: its negative), the `doosum` row scale of the reference's
// backward (flashattn_bwd_preprocess, attn_tl.py:196-221); plane 1 = lse in log2 units, the form the two
// other launches subtract inside exp2.  DV/8 lanes share a row, 16 bytes each.
//
// Bound by the read of do and o.  A workgroup has 32 positions of as many heads as a wave's load of 1 KiB spans (heads lie side by side
// in memory): a thread's 16 loads are in flight together, and a head's 32 row values leave as one line.  With one load of either
// tensor a thread, rows found by 64-bit divisions and values stored four bytes a line (before -> now, us): D128 B4 H32 S2048
// 26.9 -> 21.5 (6.2 TB/s), B8 H32 S875 23.6 -> 19.4, B5 H32 S2676 42.1 -> 35.8.
#define AE_DELTA_S 32                          // positions of a workgroup, as the host counts them
#define AE_DELTA_H (64 / (AE_DV / 8))          // heads
template <int I> struct ae_delta_ctrl { static constexpr int value = I; };
AE_DEV float ae_delta_row_sum(float x) {       // over the DV/8 lanes of a row, each with the lane 1, 2, 4, 8 away
  auto swapped = [](float v, auto ctrl) AE_LAMBDA -> float {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 15, 15, true));
  };
  x += swapped(x, ae_delta_ctrl<0xB1>());      // quad_perm 1 0 3 2
  x += swapped(x, ae_delta_ctrl<0x4E>());      // quad_perm 2 3 0 1
  x += swapped(x, ae_delta_ctrl<0x141>());     // row_half_mirror: the other four of eight, which are alike
  if (AE_DV == 128) x += swapped(x, ae_delta_ctrl<0x140>());     // row_mirror
  return x;
}
extern "C" __global__ __launch_bounds__(256)
void ae_bwd_delta_kernel(const ae_attn_bwd_params p) {
  constexpr int LPR = AE_DV / 8, NI = AE_DELTA_S / 4;      // lanes a row; positions of a wave
  __shared__ float sums[AE_DELTA_H][AE_DELTA_S];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n_hg = (p.heads_q + AE_DELTA_H - 1) / AE_DELTA_H, n_sc = (p.seqlen_q + AE_DELTA_S - 1) / AE_DELTA_S;
  int hg, sc;
  const int b = ae_divide(ae_divide(blockIdx.x, n_hg, hg), n_sc, sc);
  const int h0 = hg * AE_DELTA_H, s0 = sc * AE_DELTA_S;
  // the row value that this thread writes: its lse comes with the rows
  const int wh = tid / AE_DELTA_S, ws = tid % AE_DELTA_S;
  const bool writes = tid < AE_DELTA_H * AE_DELTA_S && h0 + wh < p.heads_q && s0 + ws < p.seqlen_q;
  const int64_t plane = (int64_t)p.batch * p.heads_q * p.seqlen_q;
  const int64_t ri = ((int64_t)b * p.heads_q + h0 + wh) * p.seqlen_q + s0 + ws;
  const float l = p.lse && writes ? p.lse[ri] : 0.f;
  {
    // (heads and positions past the end read the last one)
    const int h = h0 + lane / LPR < p.heads_q ? h0 + lane / LPR : p.heads_q - 1, c = lane % LPR * 8;
    const ae_elem* o = (const ae_elem*)p.out + (int64_t)b * p.o_stride_b + (int64_t)h * p.o_stride_h + c;
    const ae_elem* d = (const ae_elem*)p.dout + (int64_t)b * p.do_stride_b + (int64_t)h * p.do_stride_h + c;
    ae_elem8 ov[NI], dv[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
      int s = s0 + wave * NI + i;
      s = s < p.seqlen_q ? s : p.seqlen_q - 1;
      ov[i] = *(const ae_elem8*)(o + (int64_t)s * p.o_stride_s);
      dv[i] = *(const ae_elem8*)(d + (int64_t)s * p.do_stride_s);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NI; i++) {
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j++) acc += (float)ov[i][j] * (float)dv[i][j];
      acc = ae_delta_row_sum(acc);
      if (lane % LPR == 0) sums[lane / LPR][wave * NI + i] = acc;
    }
  }
  __syncthreads();
  if (writes) {
    const float acc = sums[wh][ws];
#if AE_BWD_KIND == 0
    p.delta[ri] = -acc;             // (the sign in which the two launches start their dp products)
#else
    p.delta[ri] = acc;
#endif
#if AE_BWD_KIND == 2
    // further planes: the online function's final row scales, as the forward wrote them
    p.delta[plane + ri] = l;
#pragma unroll
    for (int i = 1; i < AE_BWD_NRS; i++) p.delta[(1 + i) * plane + ri] = p.more_rowscales[i - 1][ri];
#else
    // second plane: lse in log2 units, +inf for a row without a visible key (its p is 0 everywhere)
    p.delta[plane + ri] = (l == AE_NEG_INF) ? __builtin_inff() : l * AE_LOG2E;
#endif
  }
}

#endif
