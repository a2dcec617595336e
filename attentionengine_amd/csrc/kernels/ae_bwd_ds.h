// ds of a softmax backward in memory, as the dk/dv launch (ae_prefill_bwd.hip, AE_BWD_KEEP_DS) leaves it for the dq launch
// (ae_bwd_dq.hip): for every (batch, q head), q tile of 64 rows and 32 keys a block of 4 KiB, in the operand layout in which
// the wave that forms it holds it - [k-step kk of 16 q rows][lane][8 values of 16 bits]: lane 32*hf + l has key l and, in slots
// j, the q rows 16*kk + 8*(j/4) + 4*hf + j%4.  A q tile's blocks are contiguous, in the order of the keys.  Under a causal mask
// over equal lengths only the blocks that hold something visible exist (those of 128-key tiles up to the diagonal).  All of it
// lies in the work buffer, behind its two planes.
// Needs AE_MASK_MODE.

#ifndef AE_BWD_DS_H
#define AE_BWD_DS_H

// pairs of blocks (64 keys) of q tile tq
AE_DEV int ae_ds_pairs(const ae_attn_bwd_params& p, int tq) {
  if (AE_MASK_MODE == 1 && p.seqlen_q == p.seqlen_kv) return 2 * (tq / 2 + 1);
  return 2 * ((p.seqlen_kv + 127) / 128);
}
// ... of the q tiles in front of tq
AE_DEV int ae_ds_pairs_before(const ae_attn_bwd_params& p, int tq) {
  if (AE_MASK_MODE == 1 && p.seqlen_q == p.seqlen_kv) return 2 * (tq / 2) * (tq / 2 + 1) + (tq & 1) * 2 * (tq / 2 + 1);
  return tq * (2 * ((p.seqlen_kv + 127) / 128));
}
// first block of q tile tq of (batch, q head) bh
AE_DEV char* ae_ds_row(const ae_attn_bwd_params& p, int bh, int tq) {
  const int64_t planes = ((int64_t)2 * p.batch * p.heads_q * p.seqlen_q + 3) & ~(int64_t)3;
  return (char*)(p.delta + planes) + ((int64_t)bh * ae_ds_pairs_before(p, (p.seqlen_q + 63) / 64) + ae_ds_pairs_before(p, tq)) * 8192;
}

#endif
