// The row sums that a backward needs in front of its two launches, as a launch of its own: with AE_BWD_KIND 0 where the dq
// launch comes last (ae_bwd_dq.hip), for the other kinds always.  Needs AE_DV, AE_BWD_KIND, AE_BWD_NRS.

#ifndef AE_BWD_DELTA_H
#define AE_BWD_DELTA_H

// Work buffer fp32 [2,B,Hq,Sq]: plane 0 = rowsum(do * o) (softmax: its negative), the `doosum` row scale of the reference's
// backward (flashattn_bwd_preprocess, attn_tl.py:196-221); plane 1 = lse in log2 units, the form the two
// other launches subtract inside exp2.  DV/8 lanes share a row, 16 bytes each.
extern "C" __global__ __launch_bounds__(256)
void ae_bwd_delta_kernel(const ae_attn_bwd_params p) {
  constexpr int LPR = AE_DV / 8;                   // lanes per row
  constexpr int RPB = 256 / LPR;                   // rows per workgroup
  const int tid = threadIdx.x;
  const int64_t n_rows = (int64_t)p.batch * p.seqlen_q * p.heads_q;
  const int64_t row = (int64_t)blockIdx.x * RPB + tid / LPR;
  const int c = tid % LPR;
  float acc = 0.f;
  int b = 0, s = 0, h = 0;
  if (row < n_rows) {
    h = (int)(row % p.heads_q);
    s = (int)((row / p.heads_q) % p.seqlen_q);
    b = (int)(row / ((int64_t)p.heads_q * p.seqlen_q));
    const ae_elem8 o = *(const ae_elem8*)((const ae_elem*)p.out + (int64_t)b * p.o_stride_b + (int64_t)s * p.o_stride_s + (int64_t)h * p.o_stride_h + c * 8);
    const ae_elem8 d = *(const ae_elem8*)((const ae_elem*)p.dout + (int64_t)b * p.do_stride_b + (int64_t)s * p.do_stride_s + (int64_t)h * p.do_stride_h + c * 8);
#pragma unroll
    for (int j = 0; j < 8; j++) acc += (float)o[j] * (float)d[j];
  }
  // the LPR lanes of a row are consecutive and aligned: butterfly inside the group
#pragma unroll
  for (int m = 1; m < LPR; m <<= 1) {
    const int lane = tid & 63;
    acc += __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ m) << 2, __builtin_bit_cast(int, acc)));
  }
  if (row < n_rows && c == 0) {
    const int64_t ri = ((int64_t)b * p.heads_q + h) * p.seqlen_q + s;
    const float l = p.lse ? p.lse[ri] : 0.f;
#if AE_BWD_KIND == 0
    p.delta[ri] = -acc;             // (the sign in which the two launches start their dp products)
#else
    p.delta[ri] = acc;
#endif
#if AE_BWD_KIND == 2
    // further planes: the online function's final row scales, as the forward wrote them
    p.delta[(int64_t)p.batch * p.heads_q * p.seqlen_q + ri] = l;
#pragma unroll
    for (int i = 1; i < AE_BWD_NRS; i++)
      p.delta[(int64_t)(1 + i) * p.batch * p.heads_q * p.seqlen_q + ri] = p.more_rowscales[i - 1][ri];
#else
    // second plane: lse in log2 units, +inf for a row without a visible key (its p is 0 everywhere)
    p.delta[(int64_t)p.batch * p.heads_q * p.seqlen_q + ri] = (l == AE_NEG_INF) ? __builtin_inff() : l * AE_LOG2E;
#endif
  }
}

#endif
