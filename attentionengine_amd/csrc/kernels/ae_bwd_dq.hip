// dq of a softmax backward from ds in memory, for gfx950 / CDNA4: dq = ds K * scale.
//
// Role of the dq part of the reference's backward kernel (attention_engine/core/template/tl_template/attn/attn_tl.py:238-420,
// whose kv-owning workgroups add their dq contributions with fp32 atomics).  ae_prefill_bwd.hip's dq launch (AE_BWD_ROLE 0)
// forms s, dp and ds once more; where the dk/dv launch leaves its ds in memory (AE_BWD_KEEP_DS, layout: ae_bwd_ds.h) one product of
// three is left: 5 tile products a backward instead of 7, still without atomics and in a fixed order, on the same 16-bit ds.
//
// Bound by memory: 16 KiB of ds and 8 KiB of K a step of 32 keys, for 8 MFMAs a wave.  A workgroup owns 256 q rows of a (batch,
// q head), a wave 32 of them; two workgroups share a CU.  OUT^T[d, q] += K^T[d, kv] ds^T[kv, q] with v_mfma_f32_32x32x16: both operands come
// out of LDS through ds_read_b64_tr_b16 in the same order of the keys, K as in ae_prefill_bwd.hip, ds as a tile of 32 keys x
// 64 slots of q rows a q tile (a wave uses 32 of the slots; where slot n lies among the rows is undone when the rows leave).
// Three stages of 24 KiB, filled by direct loads two steps ahead.
//
// B4 H32 S2048 D128 bf16 causal (570 MB of ds, 812 MB moved): 141 us, 5.8 TB/s, where the launch that forms ds takes 219.  One workgroup
// a CU 160 at first, two 152 with the steps from the last keys to the first, past the caches 145 (loads that stay in them: 150 for 141).
// Loads whose neighbouring lanes read neighbouring bytes, us, before and after: that call 149 -> 141, fp16 B2 H32 S4096 247 -> 235, bf16 B8
// H32 S875 84.7 -> 77.3, B5 Hq32 Hkv8 S2676 289 -> 259.  With all of ds in the L2 it would be 90.  Heads four or eight at a time, so that
// their K stays in the L2: 150, 148 for 141; for one batch entry at a time, so that ds stays in the memory-side cache, the longest
// workgroup of each launch costs more than it saves (the backward 573 us against 538).
//
// Configuration ("ae_config.h"): AE_D (128) AE_DTYPE_BF16 AE_MASK_MODE (0, 1) AE_SM_SCALE, and for the delta kernel AE_DV AE_BWD_KIND (0).

#include "ae_hip.h"
#include "ae_config.h"
#include "ae_device.h"
#ifndef AE_BWD_NRS
#define AE_BWD_NRS 1
#endif
#include "ae_bwd_ds.h"
#include "ae_bwd_delta.h"

#define AE_NWAVES 8
#define AE_BR (AE_NWAVES * 32)     // q rows per workgroup
#define AE_BS 32                   // keys per step
#define AE_STR (AE_D * 2)          // LDS row pitch of the K tile, bytes
#define AE_K_BYTES (AE_BS * AE_STR)
#define AE_DS_BYTES 4096           // 32 keys x 64 slots of one q tile: a block
#define AE_STAGE_BYTES (AE_K_BYTES + 4 * AE_DS_BYTES)
#define AE_NSTAGE 3
#define AE_NDB (AE_D / 32)         // 32-wide column blocks of dq
#define AE_KL (AE_K_BYTES / 1024 / AE_NWAVES)     // K loads per wave and step
#define AE_DL 2                    // ds loads per wave and step: half a block
#define AE_NKK (AE_BS / 16)        // k-steps over a step's keys
#define AE_VMCNT(n) (0x0F70 | ((n) & 15) | (((n) >> 4) << 14))
#define AE_AHEAD 4                 // LDS fragments in flight ahead of the MFMA that uses them

static_assert(AE_D == 128 && AE_DV == 128, "head dim 128");
static_assert(AE_MASK_MODE == 0 || AE_MASK_MODE == 1, "none or causal");

typedef __attribute__((address_space(3))) unsigned char ae_lds_byte;

// LDS position of 16-byte chunk c of row r of K, as in ae_prefill_bwd.hip: an involution in c
AE_DEV int ae_chunk_pos(int r, int c) { return ((((c >> 1) ^ (r & 7)) << 1) | ((c ^ (r >> 3)) & 1)); }

extern "C" __global__ __launch_bounds__(AE_NWAVES * 64) __attribute__((amdgpu_waves_per_eu(4, 4)))
void ae_bwd_dq_kernel(const ae_attn_bwd_params p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char ae_smem[];
  ae_lds_byte* lds = (ae_lds_byte*)ae_smem;       // AE_NSTAGE stages of [K tile][ds of four q tiles]
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int hf = lane >> 5;

  // ids as in ae_prefill_bwd.hip: the q tiles of a head on one XCD, under a causal mask the longest first
  const int n_rt = (p.seqlen_q + AE_BR - 1) / AE_BR;
  const int n_bh = p.batch * p.heads_q;
  const int n_bg = (n_bh + 7) >> 3;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  int turn;
  const int tile = ae_divide(slot, n_bg, turn);
  const int bh = ae_head_of_xcd(turn, xcd, n_bh, p.heads_q != p.heads_kv && n_bg >= AE_RUNS_FROM);
  const int rt = AE_MASK_MODE == 1 ? n_rt - 1 - tile : tile;
  if (bh >= n_bh) return;
  const int h = bh % p.heads_q, b = bh / p.heads_q;
  const int hk = h / (p.heads_q / p.heads_kv);
  const int r0 = rt * AE_BR;
  const int r0w = r0 + wave * 32;

  const int n_st = (p.seqlen_kv + AE_BS - 1) / AE_BS;
  int n_items = n_st, n_mine = n_st;             // steps of the workgroup, and those in which the wave's rows see a key
#if AE_MASK_MODE == 1
  n_items = (r0 + AE_BR - 1) / AE_BS + 1 < n_st ? (r0 + AE_BR - 1) / AE_BS + 1 : n_st;
  n_mine = (r0w + 31) / AE_BS + 1 < n_items ? (r0w + 31) / AE_BS + 1 : n_items;
#endif

  // ---- requests: K rows wave * 4 .. + 3 of the step's 32, and half a block of ds: 1 KiB pieces kk = 2 * (wave % 2) .. + 1 of q tile
  // wave / 2.  A piece lands as it lies in memory but for its groups of four keys (64 bytes), which are exchanged inside 256 bytes: a
  // transposed read takes four of them, of two pieces and of either half of a piece, that would share their banks.  (A load whose
  // sixteen neighbouring lanes read 32 bytes each of eight lines - ds with its rows of 64 slots side by side in LDS - is
  // held at issue: 520 to 1370 of 2800 cycles a step.)
  auto group_at = [](int kk, int half, int g) AE_LAMBDA -> int { return half * 8 + (g & 4) + ((g + 2 * half + kk) & 3); };
  const int ks = (int)p.k_stride_s;
  auto k_off = [&](int i, int back) AE_LAMBDA -> unsigned {
    const int n = (wave * AE_KL + i) * 64 + lane;
    const int r = n / 16, c = ae_chunk_pos(r, n % 16);
    const int over = r - back;                    // (rows past the end re-read the last one: their ds is zero)
    return (unsigned)(((r - (over > 0 ? over : 0)) * ks + c * 8) * 2 + 4096 - (i - AE_KL / 2) * 1024);
  };
  unsigned koff[8], doff[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    koff[i] = k_off(i < AE_KL ? i : 0, AE_BS);
    const int kk = 2 * (wave & 1) + (i < AE_DL ? i : 0), u = lane >> 2, g = (u & 4) | ((u - 2 * (u >> 3) - kk) & 3);
    doff[i] = (unsigned)(kk * 1024 + ((u >> 3) * 32 + g * 4 + (lane & 3)) * 16 + 4096 - ((i < AE_DL ? i : 0) - AE_DL / 2) * 1024);
  }
  // The steps run from the last keys to the first: the dk/dv launch goes through the key tiles from the first to the last, so
  // its last blocks are those that the memory-side cache still holds.
  const int n_qt = (p.seqlen_q + 63) / 64;
  const int tq = rt * 4 + (wave >> 1) < n_qt ? rt * 4 + (wave >> 1) : n_qt - 1;
  const int d_last = 2 * ae_ds_pairs(p, tq) - 1;       // (a q tile has blocks up to its diagonal; past them the last one is read, and not multiplied)
  int rq_x = n_items - 1;
  const char* rq_k = (const char*)((const ae_elem*)p.k + (int64_t)b * p.k_stride_b + (int64_t)hk * p.k_stride_h + (int64_t)rq_x * AE_BS * ks) - 4096;
  const char* rq_d = ae_ds_row(p, bh, tq) + (int64_t)(rq_x < d_last ? rq_x : d_last) * AE_DS_BYTES - 4096;
  auto request = [&](unsigned stage) AE_LAMBDA {
    unsigned g[8];
#pragma unroll
    for (int i = 0; i < 8; i++) g[i] = koff[i];
    if (__builtin_expect(rq_x * AE_BS + AE_BS > p.seqlen_kv, 0)) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < 8; i++) g[i] = k_off(i < AE_KL ? i : 0, p.seqlen_kv - 1 - rq_x * AE_BS);
    }
    ae_load_lds16_burst_base<AE_KL>(rq_k, g, lds + stage + (wave * AE_KL + AE_KL / 2) * 1024);
    ae_load_lds16_burst_base<AE_DL, true>(rq_d, doff, lds + stage + AE_K_BYTES + wave * (AE_DL * 1024) + (AE_DL / 2) * 1024);
    // (past the first keys they are read again: every call makes the same number of requests)
    const bool more = rq_x > 0;
    rq_k -= more ? (int64_t)AE_BS * ks * 2 : 0;
    rq_d -= more && rq_x <= d_last ? AE_DS_BYTES : 0;
    rq_x -= more ? 1 : 0;
  };

  // transposed fragments, see tr_frag of ae_prefill_bwd.hip: rows 16*kk + 4*hf + 0..3 and + 8 of column 32*db + l32
  const int t_row = 4 * hf + ((lane & 15) >> 2), t_g = l32 >> 4;
  const unsigned k_lane = (unsigned)(t_row * AE_STR + ((t_g ^ (t_row & 7)) << 5) + (((lane & 3) * 8) ^ (((t_row >> 3) & 1) * 16)));
  // (key 4*g + i of slots 16*kk + 8*half ..: group g; 8 keys on the group's low bits change by 2)
  const int d_kk = 2 * (wave & 1) + t_g, d_half = (lane & 3) >> 1;
  const unsigned d_lane = (unsigned)(AE_K_BYTES + (wave >> 1) * AE_DS_BYTES + d_kk * 1024 + group_at(d_kk, d_half, hf) * 64 +
                                     ((lane & 15) >> 2) * 16 + (lane & 1) * 8);
  auto pair_of = [](const ae_lds_byte* a_lo, const ae_lds_byte* a_hi) AE_LAMBDA -> ae_elem8 {
    ae_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) ae_s16x4*)a_lo);
    ae_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) ae_s16x4*)a_hi);
    return __builtin_bit_cast(ae_elem8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  ae_f32x16 acc[AE_NDB];               // dq^T: [column][slot of a q row]
#pragma unroll
  for (int db = 0; db < AE_NDB; db++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[db][r] = 0.f;

  request(0);
  request(AE_STAGE_BYTES);
  unsigned st_use = 0, st_req = 2 * AE_STAGE_BYTES;
  const unsigned lds0 = (unsigned)(unsigned long)lds;
  for (int x = n_items - 1; x >= 0; x--) {
    __builtin_amdgcn_s_waitcnt(AE_VMCNT(AE_KL + AE_DL));     // the step's tiles have landed, the next one's are on their way
    __syncthreads();
    request(st_req);                                         // into the stage everyone has left
    if (x < n_mine) {
      unsigned ka = lds0 + st_use + k_lane, da = lds0 + st_use + d_lane;
      asm("" : "+v"(ka), "+v"(da));
      auto k_frag = [&](int f) AE_LAMBDA -> ae_elem8 {
        const int kk = f / AE_NDB, db = f % AE_NDB;
        return pair_of((const ae_lds_byte*)(ka ^ (unsigned)(db << 6)) + kk * 16 * AE_STR,
                       (const ae_lds_byte*)(ka ^ (unsigned)((db << 6) | 16)) + (kk * 16 + 8) * AE_STR);
      };
      ae_elem8 ds[AE_NKK], ring[AE_AHEAD + 1];
#pragma unroll
      for (int kk = 0; kk < AE_NKK; kk++) ds[kk] = pair_of((const ae_lds_byte*)da + kk * 256, (const ae_lds_byte*)(da ^ 128u) + kk * 256);
#pragma unroll
      for (int f = 0; f < AE_AHEAD; f++) ring[f] = k_frag(f);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = 0; f < AE_NKK * AE_NDB; f++) {
        if (f + AE_AHEAD < AE_NKK * AE_NDB) ring[(f + AE_AHEAD) % (AE_AHEAD + 1)] = k_frag(f + AE_AHEAD);
        acc[f % AE_NDB] = ae_mfma32(ring[f % (AE_AHEAD + 1)], ds[f / AE_NDB], acc[f % AE_NDB]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    st_use = st_use == 2 * AE_STAGE_BYTES ? 0 : st_use + AE_STAGE_BYTES;
    st_req = st_req == 2 * AE_STAGE_BYTES ? 0 : st_req + AE_STAGE_BYTES;
  }
  __builtin_amdgcn_s_waitcnt(AE_VMCNT(0));             // nothing may land in LDS any more: the ring takes the rows
  __syncthreads();

  // ---- the rows leave through LDS: slot n = 8*c + j of the wave's q tile is row 16*(c/2) + 8*(j/4) + 4*(c%2) + j%4 ----------
  {
    int le = lane;
    asm volatile("" : "+v"(le));
    ae_lds_byte* os = lds + wave * (32 * AE_STR);
    const int n = le & 31, row_of = 16 * (n >> 4) + 8 * ((n >> 2) & 1) + 4 * ((n >> 3) & 1) + (n & 3);
    ae_lds_byte* orow = os + row_of * AE_STR + (le >> 5) * 8;
#pragma unroll
    for (int db = 0; db < AE_NDB; db++)
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        ae_elem4 w;
#pragma unroll
        for (int t = 0; t < 4; t++) w[t] = (ae_elem)(acc[db][rg * 4 + t] * AE_SM_SCALE);
        *(__attribute__((address_space(3))) ae_elem4*)(orow + (((db * 4 + rg) ^ (row_of & 15)) << 4)) = w;
      }
    // (the rows were written by other lanes of this wave: LDS instructions of a wave complete in order)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    ae_elem* o = (ae_elem*)p.dq + (int64_t)b * p.dq_stride_b + (int64_t)h * p.dq_stride_h;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int at = i * 64 + le, row = at / 16, c = at % 16;
      const ae_elem8 w = *(const __attribute__((address_space(3))) ae_elem8*)(os + row * AE_STR + ((c ^ (row & 15)) << 4));
      if (r0w + row < p.seqlen_q) *(ae_elem8*)(o + (int64_t)(r0w + row) * p.dq_stride_s + c * 8) = w;
    }
  }
}
