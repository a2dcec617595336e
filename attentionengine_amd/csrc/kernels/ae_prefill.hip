// Flash-style attention forward (prefill) for gfx950 / CDNA4 with direct-to-LDS tile loads.
//
// Takes the place of the reference's TileLang prefill template
// (attention_engine/core/template/tl_template/attn/attn_tl.py:76-174) and its block-sparse
// sibling (blockattn_tl.py:49-160).  Per KV tile it keeps the reference's order of operations
// (attn_tl.py:124-164): mask -> +QK^T -> score_mod -> online_func -> cast P -> rescale O ->
// O += P V, then the epilogue and the final-rowscale store.
//
// The user-defined parts arrive in "ae_config.h" / "ae_functors.h", generated from the traced
// score_mod / mask_mod / OnlineFunc graphs (head dims 64, 128, 256; value head dims 64 ... 512):
//   configuration  AE_D AE_DV AE_BN AE_NWAVES AE_DTYPE_BF16 AE_MASK_MODE AE_HAS_MASK_MOD
//                  AE_N_ROWSCALES AE_O_SCALE_ONE AE_EVEN_Q AE_EVEN_KV AE_WAVES_PER_EU
//   functors       ae_rowstate, ae_rowstate_init, ae_mask_mod, ae_score_mod, ae_online_fwd,
//                  ae_epilogue, ae_load_custom
//
// Same mapping to the matrix cores as ae_prefill_simple.hip (which documents the register layouts
// in full): S^T = K Q^T and O^T += V^T P^T with v_mfma_f32_32x32x16, one query row per lane, Q in
// registers, P handed from the first product to the second without leaving registers.
//
// What differs is how K / V tiles reach LDS.  Measured on MI355X, staging a tile through VGPRs
// (global_load -> 32 registers -> ds_write_b128) costs this kernel a third of its throughput: the
// wave issues in order, so the extra loads, the wait for them and the LDS writes all sit on the
// critical path of the two waves that share a SIMD.  Here every lane issues
// `global_load_lds_dwordx4` instead: 16 bytes go from HBM/L2 straight into LDS at
// (wave-uniform base) + lane*16, no VGPRs, no ds_write, and the only wait is one vmcnt(0) in front
// of the barrier that publishes the tile.  A direct load cannot pad rows (64 lanes fill 1 KiB
// contiguously), so bank conflicts are avoided by permuting WHICH 16-byte chunk of its row a lane
// fetches:
//     K tile: LDS chunk c' of row r holds global chunk c' ^ (r mod chunks_per_row), so the
//             ds_read_b128 of 16 consecutive rows at one d offset hits 16 different bank groups;
//     V tile: the permutation works on 32-byte pairs, (c'/2) ^ (r mod pairs_per_row), which keeps
//             the 4 rows x 32 bytes of one ds_read_b64_tr_b16 group on distinct banks.
// Tiles are double buffered: tile j+1 streams in while tile j is multiplied.

#include "ae_hip.h"
#include "ae_config.h"    // generated: the AE_* configuration macros
#ifndef AE_NSPLIT
#define AE_NSPLIT 1                // > 1: split-KV, p.num_splits fp32 partial results a row, merged by ae_combine.hip
#endif
#include "ae_device.h"
// custom inputs with a kv dimension (one element per score) are fetched a tile ahead: a lane's groups of four
// consecutive kv positions per tile
#define AE_KV_PF_GROUPS (AE_BN / 8)
// ... in a coalesced layout that each wave redistributes through AE_KV_SCRATCH bytes of LDS of its own per row block
// (builds with two waves per SIMD; with one, the 16 extra registers and the staging cost more than they save:
// retention at D 256, DV 512 0.88 against 0.78 ms)
#define AE_KV_COALESCED (AE_WAVES_PER_EU >= 2)
#define AE_KV_SCRATCH 2560
#include "ae_functors.h"  // generated: the functor bodies
#include "ae_tile_table.h"
#ifndef AE_HEAVY_LAST
#define AE_HEAVY_LAST 0      // 1: the tile table gives late q tiles more work than early ones
#endif

// AE_BAND 1 (AE_MASK_MODE 2 in the configuration): the host has shown that mask_mod is exactly
// AE_BAND_LO <= q_idx - kv_idx <= AE_BAND_HI (core/lower/mask.py: sliding windows, shifted causal masks, a causal mask
// over unequal lengths).  Such a mask needs no table and no call of ae_mask_mod: the tile range of a q tile is a
// subtraction, a tile crosses at most two edges, and an edge costs one compare with a literal and one select per
// score.  A wave none of whose rows sees a tile does not multiply it.  B2 H32 S4096 D128 fp16, window of 256, through
// the table: 127 us (2.1 TB/s); as a band: 91 us.
#ifndef AE_BAND
#define AE_BAND 0
#endif
#if AE_BAND
#undef AE_MASK_MODE
#define AE_MASK_MODE 3
#endif
#define AE_ANALYTIC (AE_MASK_MODE == 1 || AE_MASK_MODE == 3)
#if AE_MASK_MODE == 1
#define AE_BAND_LO 0
#define AE_BAND_HI 0x7fffffff
#endif

// AE_ROTATE 1 (bands with two ends): a q tile starts at the kv tile whose index is a multiple of AE_PERIOD - the most tiles that
// a q tile's band can have, so its range holds at most one - and takes the front of its range last.  A kv tile is read by the
// (AE_BM + width) / AE_BM q tiles whose bands hold it; walked from the front of each range they come to it AE_BM / AE_BN trips
// apart, by when the 64 workgroups of an XCD have pushed it out of the 4 MB L2 (20 % hits, 410 MB read for 201 MB of q, k and v).
// Started this way, workgroups in step with each other read the same tile in the same trip.  Inputs not in the caches, B2 H32
// S4096 D128 fp16: window 256 85.9 -> 76.8 us; calls one after the other, window 1024 162.4 -> 155.8, B4 S4000 bf16 window 64
// 119.8 -> 116.4, B3 S5188 bf16 window 388 179.2 -> 169.3; B1 H128 S2500 192 / 128 columns window 512 162.2 -> 142.5, sigmoid weights,
// window 256, 82.0 -> 73.4 and at 192 / 128 99.8 -> 86.2, B2 H32 S3000 160 / 128 64.9 -> 61.3 (14 launches of wide heads and of graphs
// without a softmax: 0.86 to 0.98 of the time).  Not at narrower heads: the keys and values of 64 neighbouring q
// tiles are 2 MB there and stay in the L2 anyway (B2 H16 S2886 D64 window 843 32.8 -> 33.8).
#define AE_ROTATE (AE_MASK_MODE == 3 && AE_BAND_HI != 0x7fffffff && AE_NSPLIT == 1 && AE_KW == 1 && AE_D + AE_DV >= 256)

// AE_KW > 1: the waves of a workgroup also share the kv axis.  AE_NWAVES waves own 32 query rows each, as always; AE_KW
// such sets of waves ("kv groups") walk the kv tiles in turn, each with its own pair of LDS stages, and meet at the end:
// every wave leaves its unscaled O in LDS, rescales a share of the value columns to the common reference and sums it
// over the groups.  For launches whose q tiles do not fill the chip - one prompt of a few hundred tokens, a chunk of
// query tokens against a long cache -, where a wave alone on its SIMD takes 1.5 us for a 64-key tile (LDS latency, MFMA
// latency and the softmax one after the other) and the kv axis is a serial chain of them: B1 Hq32 S333 causal, 96
// workgroups, 9.4 of 13.4 us in six tiles.  Needs a merge that the kernel knows: AE_KW_SOFTMAX 1 the proven online softmax
// (fields AE_SM_M, AE_SM_R), 0 no row state (O is summed).  Not with a tile table.
#ifndef AE_KW
#define AE_KW 1
#endif
#ifndef AE_KW_SOFTMAX
#define AE_KW_SOFTMAX 0
#endif

// K / V tiles in LDS.  2: tile j + 1 is requested at the start of trip j and waited for at its end.  3 (split launches at head
// dim 128, a workgroup a CU): tile j + 2 is, into the stage of tile j - 1, and the wait at the end is for tile j + 1 alone.  Such
// a launch is bound by the cache's bytes, and with two stages nothing is on its way from the last byte's arrival until the
// next trip.  us: B1 H32 Sq128 Skv8192 42.2 -> 39.4, B3 H32 Sq48 Skv5012 62.7 -> 52.5, B3 H32 Sq3 Skv1218 18.8 -> 17.3 (four
// stages 40.7, 53.3, 18.2).  Not where the workgroups share CUs: a sliding window B2 H32 S4096 D128 75.5 -> 74.9 (four 80.7),
// causal 192 / 128 columns 293 -> 322 (two workgroups a CU instead of three).
#ifndef AE_KV_STAGES
#define AE_KV_STAGES 2
#endif
// 1 (split builds with kv groups): where p.tail_slots is not 0 the workgroup that finishes last of a q tile merges, see
// ae_merge_last.h; p.num_splits at most 8 then
#ifndef AE_MERGE_LAST
#define AE_MERGE_LAST 0
#endif
#if AE_MERGE_LAST
#include "ae_merge_last.h"
static_assert(AE_NSPLIT > 1 && AE_KW > 1, "merged by the last workgroup: builds whose groups meet in LDS");
#endif
#define AE_DEEP (AE_KV_STAGES == 3)

// value given to score positions past seqlen_kv before the user functors run: -inf, or 0 for graphs
// declared with mask_value="0" (no additive -inf mask anywhere, attn_tl.py:124-137 / lower.py:637)
#if defined(AE_MASK_VALUE_ZERO) && AE_MASK_VALUE_ZERO
#define AE_KV_PAD 0.f
#else
#define AE_KV_PAD AE_NEG_INF
#endif

// 1: the proven online softmax - a score of -inf leaves the functor as exactly 0 (the running maximum starts at a
// finite -1e38), so keys past the end need no second test
#ifndef AE_PAD_GIVES_ZERO
#define AE_PAD_GIVES_ZERO 0
#endif
// 1: an elementwise graph (out = sum_kv f(s) v: no row state, no use of the kv index).  The weight of a key past the end is
// set to 0 whatever its score was - f(0) of a row of zeros need not be finite once it is in the input type, an infinite
// query times a row of zeros is NaN, and a V whose rows overlap (expanded along the sequence) has no rows of zeros -, so
// its score needs no test, except where the mask's own test decides whether the row has seen a key
#ifndef AE_ELEMENTWISE
#define AE_ELEMENTWISE 0
#endif
#define AE_PAD_SCORES (!AE_EVEN_KV && AE_MASK_MODE != 1 && !(AE_ELEMENTWISE && (AE_ANALYTIC || !AE_HAS_MASK_MOD)))
#define AE_PAD_WEIGHTS (!AE_EVEN_KV && !AE_PAD_GIVES_ZERO)
#ifndef AE_RB
#define AE_RB 1
#endif
// AE_OWN_SOFTMAX 1 (the proven online softmax of score * AE_SM_SCALE, fields AE_SM_M and AE_SM_R): written out here.  A row's
// reference moves where a score exceeds it by AE_SM_TAU, which a lane sees by itself: two lanes share a row, and only where some
// lane of the wave has such a score do they exchange their maxima and does anything move.  The row sum stays per lane until
// the end.  These kernels are bound by the VALU at head dim 64.  us, generated functors (which exchange maxima and sums on every
// tile) -> this, addresses by constants (below) included, at scores with a standard deviation of 1 | 4 | 16: bf16 B16 H16 S1000
// D64 86.3 -> 83.3 | 90.0 -> 88.0 | 91.7 -> 90.4, causal B2 H32/8 S3407 D64 116.1 -> 110.5 | 118.8 -> 115.2 | 120.6 -> 118.5,
// B4 H32 S1500 D128 99.6 -> 97.8 | 102.7 -> 101.5 | 104.5 -> 103.8, B1 H128 S2500 192 / 128 columns 290 -> 275 | 302 -> 290 |
// 307 -> 297.  (Without any maxima, a tile whose weights' sum is too large multiplied again: 84 | 86.7 | 119.5 for the
// first, 281 | 290 | 359 for the last; and what one row makes its wave do twice changed the rounding of the others.)
#ifndef AE_OWN_SOFTMAX
#define AE_OWN_SOFTMAX 0
#endif
#define AE_SM_TAU 5.545177444479562f     // 8 log2 units: weights up to 256
// AE_FIRST_REST 1 (split launches with kv groups whose tiles PrefillOp._cheapest_form chooses): what the rounding of its first
// tile's weights leaves over is multiplied as well.  The largest weight of every reference is 1, which has no rounding error,
// and the plans with fewer splits and kv groups have fewer references: by that alone the error against fp64 was 1.019 of what
// four groups and a split for every CU gave (40 shapes of 1 to 256 rows, 512 to 16384 keys, N(0, 1) scores; 1.08 at most), the
// more the shorter the cache.  So it is 0.990 (1.02); on 50 shapes of more than 32 rows 1.012 without, 1.000 so (1.09 at most,
// where ten splits have become one).  0.2 to 0.3 us a call; every tile's: 7 % of 60 calls of 9 to 330 us, error 0.74; the
// references that there were, by the plan: 3.5 % of calls of at most 32 rows.
#ifndef AE_FIRST_REST
#define AE_FIRST_REST 0
#endif
// 1: a wave's priority on its SIMD goes up as it goes through a trip - scores 0, softmax 1, second product 2 -, so that of the waves
// that share the SIMD the one that has got furthest finishes and they fall out of step: one's products run under another's
// softmax.  us: causal 192 / 128 columns B1 H128 S2500 278 -> 270, B2 H128 S1400 222 -> 208, B1 H32 S5000 249 -> 236, B4 H128 S700 163 ->
// 158; sigmoid at 64 columns B2 H32 S3000 175 -> 173, B4 H16 S1000 25.6 -> 24.7.  Not at 128 columns (causal B4 Hq32 Hkv8 S1400 79.2 ->
// 81.6) or for the softmax at 64 (155.5 -> 157.1), and not where the groups of a workgroup wait for each other (192 / 128 B1 H16
// S8000 315 -> 320).
#define AE_PRIO (AE_KW == 1 && AE_NSPLIT == 1 && AE_WAVES_PER_EU >= 2 && (AE_D >= 192 || (AE_ELEMENTWISE && AE_D <= 64)))
#define AE_SETPRIO(n) do { if (AE_PRIO) __builtin_amdgcn_s_setprio(n); } while (0)
#define AE_TWO_ROUNDS (AE_D <= 64 ? 256 : 128)      // workgroups of two rounds of an XCD's 32 CUs
#define AE_WROWS (AE_RB * 32)     // query rows per wave
#define AE_BM (AE_NWAVES * AE_WROWS)
#define AE_GT (AE_NWAVES * 64)     // threads of a kv group
#define AE_NT (AE_GT * AE_KW)
#define AE_NB (AE_BN / 32)        // 32-wide kv blocks per tile
#if AE_ROTATE
constexpr int ae_floor_div(int a, int b) { return a >= 0 ? a / b : -((b - 1 - a) / b); }
#define AE_PERIOD (ae_floor_div(AE_BM - 1 - (AE_BAND_LO), AE_BN) - ae_floor_div(-(AE_BAND_HI), AE_BN) + 1)
#endif
#define AE_VMCNT(n) (0x0F70 | ((n) & 15) | (((n) >> 4) << 14))
#define AE_NS (AE_NB * 16)        // score elements per lane per tile
#define AE_NDB (AE_DV / 32)       // 32-wide dv blocks
#define AE_NO (AE_NDB * 16)       // output elements per lane
#define AE_KSTR (AE_D * 2)        // LDS row pitch of the K tile, bytes (no padding: swizzled)
#define AE_VSTR (AE_DV * 2)       // LDS row pitch of the V tile, bytes
#define AE_K_BYTES (AE_BN * AE_KSTR)
#define AE_V_BYTES (AE_BN * AE_VSTR)
#define AE_STAGE_BYTES (AE_K_BYTES + AE_V_BYTES)
#define AE_KCPR (AE_D / 8)        // 16-byte chunks per K row
#define AE_VCPR (AE_DV / 8)
#define AE_K_LOADS ((AE_BN * AE_KCPR) / AE_GT)   // direct loads per lane per K tile
#define AE_V_LOADS ((AE_BN * AE_VCPR) / AE_GT)
#define AE_V_RPI (64 / AE_VCPR)
#define AE_KGRP ((AE_KCPR & (AE_KCPR - 1)) == 0 ? AE_KCPR : (AE_KCPR % 16 == 8 ? 8 : 4))    // chunks that ae_k_swz exchanges
#define AE_VPPR (AE_VCPR / 2)     // 32-byte pairs per V row
// the pairs of a V row are exchanged by the row's low bits: at most three of them, so that rows 8 apart (the
// two halves of a transposed fragment) share one permutation whatever the row length
#define AE_VSWM ((AE_VPPR < 8 ? AE_VPPR : 8) - 1)

static_assert(AE_D % 16 == 0, "head dim must be a multiple of 16");
static_assert(AE_DV % 32 == 0, "value head dim must be a multiple of 32");
static_assert(AE_BN % 32 == 0, "kv tile must be a multiple of 32");
static_assert((AE_BN * AE_KCPR) % AE_GT == 0, "K tile must split evenly over the waves that load it");
static_assert((AE_BN * AE_VCPR) % AE_GT == 0, "V tile must split evenly over the waves that load it");
static_assert(AE_KW == 1 || (AE_MASK_MODE != 2 && AE_RB == 1 && AE_NO % (4 * AE_KW) == 0 && AE_WAVES_PER_EU >= 2),
              "kv groups: 32 rows a wave, no tile table, a whole number of 4-column pieces of O per group");
static_assert(AE_KV_STAGES == 2 || (AE_DEEP && AE_MASK_MODE == 0), "two or three stages; tiles requested ahead follow one another");
static_assert(AE_K_LOADS >= 1 && AE_K_LOADS <= 8 && AE_V_LOADS >= 1 && AE_V_LOADS <= 8, "one burst per tile and wave");
static_assert(AE_KCPR == 8 || AE_KCPR == 16 || AE_KCPR == 32 || AE_KCPR % 8 == 4 || AE_KCPR % 16 == 8,
              "swizzle is written for K rows of 128, 256 or 512 bytes, or an odd multiple of 64 or 128 bytes");
static_assert(AE_VCPR == 8 || AE_VCPR == 16 || AE_VCPR == 32 || AE_VCPR == 64, "swizzle is written for 128- to 1024-byte V rows");

typedef __attribute__((address_space(3))) unsigned char ae_lds_byte;
template <bool B> struct ae_const_bool { static constexpr bool value = B; };

// LDS chunk of K row `row` that holds global chunk c (and the other way round: an involution).  A fragment read
// (ds_read_b128) takes one chunk index of 16 consecutive rows; they must fall into 16 different groups of four
// banks.  Rows of a power-of-two length all start in the same group, so the chunk index is exchanged by the row
// number.  Rows of 8*odd chunks (head dim 192: 384 bytes) start in two alternating groups and rows of 4*odd
// chunks (head dims 96, 160) in four, so only the low three (two) bits of the chunk index are exchanged, by the
// row number without the bits that the row pitch already spreads.
AE_DEV int ae_k_swz(int c, int row) {
#if (AE_KCPR & (AE_KCPR - 1)) == 0
  return c ^ (row & (AE_KCPR - 1));
#elif AE_KCPR % 16 == 8
  return c ^ ((row >> 1) & 7);
#else
  return c ^ ((row >> 2) & 3);
#endif
}

// Fragments that a wave reads from LDS ahead of the MFMA that takes them: rings with one scheduling fence per MFMA (left
// to itself the compiler keeps one or two reads in flight and waits for each).  Not in the builds that run one wave per SIMD
// with every register taken.  bf16, without a mask, B16 H16 S1000: D 64 90.0 -> 88.2 us, D 128 160.3 -> 155.6 us (with the
// shorter epilogue); causal B8 H32 S1000 D128 112.3 -> 110.0 us.  At D 192, DV 128 the rings have cost a wave per SIMD (180
// registers, 294 -> 313 us); without row maxima and with fragment addresses by constants 168 suffice: B1 H128 S2500 299.6 ->
// 290.0, B1 H16 S8088 345 -> 329, B2 H32 S1968 105.9 -> 101.5, B1 H32 S570 16.5 -> 15.8, B3 H16 S789 26.7 -> 27.1 (24.8 with AE_OWN_SOFTMAX as well; rings of
// two and two, three and three, six and three fragments: 289.8, 291.0, 305.7 for the first; none 280 to 288 there, 44.7
// against 42.8 for B2 H32 S1098).  At D 160 fragment addresses by constants without the rings cost up to 9 % (B4 H16 S1000 causal
// 36.4 -> 38.1, B1 H32 S333 14.1 -> 15.0), with them 192 calls (DV 64 and 128, softmax, sigmoid and relu, every kind of mask) take
// 0.92 of the time before either, none more than 1.01: 33.1 and 12.7 for those two.
#if AE_D <= 192 && AE_DV <= 128 && AE_RB == 1
#define AE_K_AHEAD 4
#define AE_V_AHEAD 3
#define AE_RING_FENCE() __builtin_amdgcn_sched_barrier(0)
#else
#define AE_K_AHEAD 0
#define AE_V_AHEAD 0
#define AE_RING_FENCE()
#endif

// Q rows on their way in and O rows on their way out pass through LDS as whole rows (16 lanes per 256-byte row).
// A lane that loads its own row's fragments, or stores its own row's results, touches 32 rows per instruction,
// 16 bytes of each: the workgroups of a launch start and end together and queue behind each other's requests
// (measured in the pipelined kernel: 3.5 us until the first tile could be multiplied, 4.4 us to get O out).
// Q uses the last stage of the tile ring, which is free until the loop's first prefetch, swizzled like a K tile; O the
// whole ring after the last tile.  Builds whose rows do not fit there keep the direct accesses.
#define AE_Q_LOADS ((AE_WROWS * AE_KCPR) / 64)     // direct loads per lane for the wave's Q rows
#define AE_Q_VIA_LDS (AE_BM * AE_KSTR <= AE_STAGE_BYTES)
#define AE_O_LOADS ((AE_WROWS * AE_VCPR) / 64)
#define AE_O_VIA_LDS (AE_NSPLIT == 1 && AE_KW == 1 && AE_NO <= 128 && AE_BM * AE_VSTR <= 2 * AE_STAGE_BYTES)

// the wave's Q rows -> qs, in bursts of up to eight loads.  qg: row q0c of this (batch, head), 4 KiB low (see
// ae_load_lds16_burst_base); row0 = first row of the wave - q0c; rows past `last` (relative to q0c) re-read it.
template <int G0>
AE_DEV void ae_q_rows_to_lds(const char* qg, ae_lds_byte* qs, int lane, int row0, int last, int stride_s) {
  if constexpr (G0 < AE_Q_LOADS) {
    constexpr int N = AE_Q_LOADS - G0 < 8 ? AE_Q_LOADS - G0 : 8;
    unsigned off[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int n = (G0 + (i < N ? i : 0)) * 64 + lane;      // chunk of the wave's rows, in LDS order
      const int row = n / AE_KCPR;
      const int c = ae_k_swz(n % AE_KCPR, row);
      int ra = row0 + row;
      ra = ra < last ? ra : last;
      off[i] = (unsigned)((ra * stride_s + c * 8) * 2 + 4096 - (i - N / 2) * 1024);
    }
    ae_load_lds16_burst_base<N>(qg, off, qs + (G0 + N / 2) * 1024);
    ae_q_rows_to_lds<G0 + 8>(qg, qs, lane, row0, last, stride_s);
  }
}

extern "C" __global__ __launch_bounds__(AE_NT)
__attribute__((amdgpu_waves_per_eu(AE_WAVES_PER_EU)))
void ae_prefill_kernel(const ae_attn_params p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char ae_smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
#if AE_KW == 1
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  ae_lds_byte* lds = (ae_lds_byte*)ae_smem;
#else
  const int wave_wg = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave_wg / AE_NWAVES;         // kv group
  const int wave = wave_wg % AE_NWAVES;       // ... and which 32 rows
  ae_lds_byte* lds = (ae_lds_byte*)ae_smem + kg * (AE_KV_STAGES * AE_STAGE_BYTES);
#endif
  const int l32 = lane & 31;
  const int hf = lane >> 5;

  // ---- which (q-tile, head, batch) -----------------------------------------------------
  // The dispatcher deals consecutive workgroup ids round-robin to the 8 XCDs, each with its own
  // L2.  All q-tiles of one (batch, head) read the same K/V, so they are given ids that land on
  // ONE XCD back to back (id = 8*slot + xcd, slot = bh_local*n_qt + qt_i): the tiles run
  // concurrently, walk the kv axis roughly in step and share K/V through that XCD's L2.
  // With a causal mask the tiles with the most kv work (last q-tiles) are issued first.
  // The grid is padded to 8*ceil(n_bh/8)*n_qt ids; surplus workgroups exit immediately.
  // (All arguments that the requests of the first tile need are read here, in one trip to memory: where they are first
  // used the compiler reads them in three, each waited for, with the arithmetic of the ids between them.)
  asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.batch), "s"(p.heads_q), "s"(p.heads_kv), "s"(p.seqlen_q),
               "s"(p.seqlen_kv), "s"(p.q_stride_b), "s"(p.q_stride_s), "s"(p.q_stride_h));
  asm volatile("" ::"s"(p.k_stride_b), "s"(p.k_stride_s), "s"(p.k_stride_h), "s"(p.v_stride_b), "s"(p.v_stride_s),
               "s"(p.v_stride_h));
  const int n_qt = (p.seqlen_q + AE_BM - 1) / AE_BM;
  const int n_bh = p.batch * p.heads_q;
#if AE_NSPLIT > 1
  // split-KV ("decode" with several query tokens): consecutive ids are the splits of one q tile
  const int n_split = p.num_splits;
  int split;
  const int wg = ae_divide(blockIdx.x, n_split, split);
#else
  const int wg = blockIdx.x;
#endif
  const int xcd = wg & 7;
  const int slot = wg >> 3;
#if AE_MASK_MODE == 1 || AE_HEAVY_LAST
  // causal: q tiles differ in work by up to n_qt : 1, so ids go heaviest tile first across ALL heads
  // (longest-job-first keeps the tail short); the heads of one XCD still meet in its L2.  A tile table whose
  // late q tiles are the long ones (AE_HEAVY_LAST, found on the host: causal variants, long sliding windows)
  // takes the same order: B2 H32 S4096, "kv <= q + 1": 0.40 -> 0.35 ms.
  int turn;
  const int n_bg = (n_bh + 7) >> 3;
  const bool own_kv = p.heads_q == p.heads_kv;
  const int n_tiles = n_bg * n_qt;
  const int qt = n_qt - 1 - ae_heavy_first(slot, n_bg, n_qt, AE_NSPLIT == 1 && AE_KW == 1 && own_kv && n_bg > 8 && n_tiles > AE_TWO_ROUNDS &&
                                           n_tiles < 1 << 22, turn);
  const int bh = ae_head_of_xcd(turn, xcd, n_bh, AE_NSPLIT == 1 && !own_kv && n_bg >= AE_RUNS_FROM);
#else
  int qt;
  const int turn = ae_divide(slot, n_qt, qt);
  const int bh = ae_head_of_xcd(turn, xcd, n_bh, AE_NSPLIT == 1 && p.heads_q != p.heads_kv && n_bh >= 8 * AE_RUNS_FROM);
#endif
  if (bh >= n_bh) return;
  int h, rest;
  const int b = ae_divide(bh, p.heads_q, h);
  const int hk = p.heads_q == p.heads_kv ? h : ae_divide(h, ae_divide(p.heads_q, p.heads_kv, rest), rest);
  const int q0 = qt * AE_BM;
  const int q0w = q0 + wave * AE_WROWS;       // first row of this wave
  int qrow[AE_RB];                             // this lane's row in each row block
  bool q_ok[AE_RB];
#pragma unroll
  for (int rb = 0; rb < AE_RB; rb++) {
    qrow[rb] = q0w + rb * 32 + l32;
#if AE_EVEN_Q
    q_ok[rb] = true;
#else
    q_ok[rb] = qrow[rb] < p.seqlen_q;
#endif
  }

  // ---- Q fragments: B operand of S^T = K Q^T, resident for the whole kernel -------------
  ae_elem8 qf[AE_RB][AE_D / 16];
#if AE_Q_VIA_LDS
  ae_lds_byte* qs = lds + (AE_KV_STAGES - 1) * AE_STAGE_BYTES + wave * (AE_WROWS * AE_KSTR);
  {
    const int q0c = q0w < p.seqlen_q ? q0w : p.seqlen_q - 1;
    const char* qg = (const char*)((const ae_elem*)p.q + (int64_t)b * p.q_stride_b + (int64_t)q0c * p.q_stride_s +
                                   (int64_t)h * p.q_stride_h) - 4096;
    ae_q_rows_to_lds<0>(qg, qs, lane, q0w - q0c, p.seqlen_q - 1 - q0c, (int)p.q_stride_s);
  }
#else
#pragma unroll
  for (int rb = 0; rb < AE_RB; rb++) {
    const int qr = q_ok[rb] ? qrow[rb] : p.seqlen_q - 1;
    const ae_elem* qptr = (const ae_elem*)p.q + (int64_t)b * p.q_stride_b +
                          (int64_t)qr * p.q_stride_s + (int64_t)h * p.q_stride_h;
#pragma unroll
    for (int ks = 0; ks < AE_D / 16; ks++) qf[rb][ks] = *(const ae_elem8*)(qptr + ks * 16 + hf * 8);
  }
#endif

  // ---- KV tile range ---------------------------------------------------------------------
  const int n_kvt = (p.seqlen_kv + AE_BN - 1) / AE_BN;
  int j_end = n_kvt;
#if AE_ANALYTIC
  int j_first = 0;        // first tile with a key that some row of the q tile sees
  {
    int last_kv = q0 + AE_BM - 1 - AE_BAND_LO;   // attn_tl.py:113-115
    last_kv = last_kv < p.seqlen_kv ? last_kv : p.seqlen_kv - 1;
    j_end = last_kv < 0 ? 0 : last_kv / AE_BN + 1;
#if AE_BAND_HI != 0x7fffffff
    const int first_kv = q0 - AE_BAND_HI;
    j_first = first_kv > 0 ? first_kv / AE_BN : 0;
#endif
  }
#endif
#if AE_MASK_MODE == 2
  // Tile classes from the block table (ae_tile_table.h): 0 = skip, 1 = visit with the elementwise mask (every
  // position, where the graph has no mask_mod: a block mask of the user), 2 = fully visible.  A q tile may span
  // several table rows: a kv tile is skipped only if every row says so, and every lane applies the class of
  // its own row.
  ae_tile_table tt;
  ae_tt_init(tt, p, b, h, q0, AE_BM);
#endif

  const ae_elem* kbase = (const ae_elem*)p.k + (int64_t)b * p.k_stride_b + (int64_t)hk * p.k_stride_h;
  const ae_elem* vbase = (const ae_elem*)p.v + (int64_t)b * p.v_stride_b + (int64_t)hk * p.v_stride_h;

  // Direct HBM -> LDS tile load.  Wave w, instruction i covers the 64 consecutive 16-byte chunks
  // (w*LOADS + i)*64 ... of the tile (whole rows when the row length is a power of two); lane L lands in LDS
  // chunk c' of row r, (w*LOADS + i)*64 + L = r*CPR + c', and fetches the permuted global chunk.
  // A lane's byte offset inside a tile never changes, so it is computed once; per tile only a
  // wave-uniform base moves.  The K loads and the V loads of a wave each go out as one burst (two beyond four loads)
  // behind a single write of M0 (ae_load_lds16_burst_rows).
  auto k_lane_off = [&](int i) AE_LAMBDA -> unsigned {
    const int chunk = (wave * AE_K_LOADS + i) * 64 + lane;     // of the tile, in LDS order
    const int row = chunk / AE_KCPR;
    const int c = ae_k_swz(chunk % AE_KCPR, row);
    return (unsigned)((row * (int)p.k_stride_s + c * 8) * 2 + 4096 - (i & 3) * 1024);
  };
  auto v_lane_off = [&](int i) AE_LAMBDA -> unsigned {
    const int row = (wave * AE_V_LOADS + i) * AE_V_RPI + lane / AE_VCPR;
    const int cp = lane % AE_VCPR;
    const int c = (((cp >> 1) ^ (row & AE_VSWM)) << 1) | (cp & 1);
    return (unsigned)((row * (int)p.v_stride_s + c * 8) * 2 + 4096 - (i & 3) * 1024);
  };
  unsigned koff[AE_K_LOADS], voff[AE_V_LOADS];
#pragma unroll
  for (int i = 0; i < AE_K_LOADS; i++) koff[i] = k_lane_off(i);
#pragma unroll
  for (int i = 0; i < AE_V_LOADS; i++) voff[i] = v_lane_off(i);
  auto load_tile = [&](int j, int stage) AE_LAMBDA {
    ae_lds_byte* ks = lds + stage * AE_STAGE_BYTES;
    ae_lds_byte* vs = ks + AE_K_BYTES;
    const char* gk = (const char*)kbase + (int64_t)j * AE_BN * p.k_stride_s * 2 - 4096;
    const char* gv = (const char*)vbase + (int64_t)j * AE_BN * p.v_stride_s * 2 - 4096;
    int rows = AE_BN;
#if !AE_EVEN_KV
    rows = p.seqlen_kv - j * AE_BN;                            // rows past the end arrive as zeros
    rows = __builtin_amdgcn_readfirstlane(rows < AE_BN ? rows : AE_BN);
    asm("" : "+s"(rows));                                      // (opaque: the compiler would split the loop over it)
#endif
    ae_load_lds16_burst_rows<AE_K_LOADS>(gk, (unsigned)(((rows - 1) * (int)p.k_stride_s + AE_D) * 2), koff,
                                         ks + wave * AE_K_LOADS * 1024);
    ae_load_lds16_burst_rows<AE_V_LOADS>(gv, (unsigned)(((rows - 1) * (int)p.v_stride_s + AE_DV) * 2), voff,
                                         vs + wave * AE_V_LOADS * 1024);
  };
  // next tile index >= j that has work (block table) or j itself
  auto next_tile = [&](int j) AE_LAMBDA {
#if AE_MASK_MODE == 2
    j = ae_tt_next(tt, p, j, j_end, AE_BN, n_kvt);
#endif
    return j;
  };
  // class of tile j for this lane's row of row block rb (right after next_tile() found j)
  auto row_class = [&](int j, int rb) AE_LAMBDA -> int {
#if AE_MASK_MODE == 2
    return j < j_end ? ae_tt_class(tt, p, j, qrow[rb]) : 0;
#else
    return 2;
#endif
  };

  // ---- state ------------------------------------------------------------------------------
  ae_ctx ctx[AE_RB];
  ae_custom cust[AE_RB];
  ae_rowstate st[AE_RB];
  ae_f32x16 oacc[AE_RB][AE_NDB];
#pragma unroll
  for (int rb = 0; rb < AE_RB; rb++) {
    ctx[rb].b = b;
    ctx[rb].h = h;
    ctx[rb].q_idx = qrow[rb];
    ctx[rb].kv_base = 0;
    ae_load_custom(cust[rb], p, ctx[rb]);
    ae_rowstate_init(st[rb]);
#pragma unroll
    for (int db = 0; db < AE_NDB; db++)
#pragma unroll
      for (int r = 0; r < 16; r++) oacc[rb][db][r] = 0.f;
  }

  // Lane parts of the LDS read addresses.  The k-step and the column block only flip bits of the chunk (pair) index inside the
  // group of chunks that the swizzle exchanges, and stages and rows start on multiples of it, so a fragment's address is
  // ((stage + lane part) ^ constant) + immediate: an addition a tile and an instruction per constant.  (From the chunk
  // positions as they are the compiler forms every address by additions: 35 of the 160 VALU instructions of a tile at head dim 64.)
  // K fragment (row l32 of a 32-row block, d chunk 2*ks+hf): see ae_k_swz
  const unsigned k_lane = (unsigned)(l32 * AE_KSTR + (ae_k_swz(hf, l32) << 4));
  // V transpose read: lane i of a 16-lane group reads row 4*hf + i/4 (+8), 8 bytes at pair
  // (2*db + g) ^ (row mod PPR), g = (lane%32)/16; rows of one group differ only in their low bits
  const int v_row = 4 * hf + ((lane & 15) >> 2);
  const unsigned v_lane = (unsigned)(v_row * AE_VSTR + (lane & 3) * 8 + (((l32 >> 4) ^ (v_row & AE_VSWM)) << 5));
  static_assert(AE_STAGE_BYTES % (AE_KGRP * 16) == 0 && AE_K_BYTES % ((AE_VSWM + 1) * 32) == 0 && AE_KSTR % (AE_KGRP * 16) == 0 &&
                AE_STAGE_BYTES % ((AE_VSWM + 1) * 32) == 0, "the exchanged bits of a stage's and a row's address are zero");

#if AE_NSPLIT > 1
  // this workgroup's share of the kv axis: kv_per_split positions (a multiple of the tile)
  const int j_begin = split * (p.kv_per_split / AE_BN);
  {
    const int lim = j_begin + p.kv_per_split / AE_BN;
    j_end = lim < j_end ? lim : j_end;
  }
#if AE_ANALYTIC
  int j = j_begin > j_first ? j_begin : j_first;
#else
  int j = next_tile(j_begin);
#endif
#elif AE_ROTATE
  int j = (j_first + AE_PERIOD - 1) / AE_PERIOD * AE_PERIOD;
  j = j < j_end ? j : j_first;
#elif AE_ANALYTIC
  int j = j_first;
#else
  int j = next_tile(0);
#endif
  bool any_tile = j < j_end;
#if AE_KW > 1
  // group kg takes tiles j0 + kg, j0 + kg + AE_KW, ...; all groups make the same number of trips (the barriers)
  const int j_trips = j_end + kg;
  j += kg;
#define AE_J_LIVE (j < j_end)
#else
  const int j_trips = j_end;
#define AE_J_LIVE true
#endif
#if AE_DEEP
  int rq_j = j, rq_stage = 0;          // the group's next tile to request, and the stage it goes into
  auto request_next = [&]() AE_LAMBDA {
    if (rq_j < j_end) load_tile(rq_j, rq_stage);
    rq_j += AE_KW;
    rq_stage = rq_stage == 2 ? 0 : rq_stage + 1;
  };
  // tile jt has landed: the one behind it, if there is one, is the only one outstanding
  auto wait_tile = [&](int jt) AE_LAMBDA {
    if (jt + AE_KW < j_end) __builtin_amdgcn_s_waitcnt(AE_VMCNT(AE_K_LOADS + AE_V_LOADS));
    else __builtin_amdgcn_s_waitcnt(AE_VMCNT(0));
  };
#endif
#if AE_ROTATE
  int left = j_end - j_first;          // tiles still to be multiplied
#endif
#if AE_ROTATE
#define AE_TRIPS_LEFT (left > 0)
#define AE_HAS_NEXT (left > 1)
#else
#define AE_TRIPS_LEFT (j < j_trips)
#define AE_HAS_NEXT (jn < j_end)
#endif
  int cls[AE_RB];          // class of tile j for this lane's row of each row block
  // 1 once this lane's row of a row block has met a key it may see.  A row that never does - inside a q tile whose
  // other rows do: block masks finer than the q tile, masks such as q - 100 >= kv - ends with out = 0 and row
  // scales of -inf, like the rows of a q tile without any tile (not with the 0 / 0 its epilogue would make of it)
  float seen[AE_RB];
#pragma unroll
  for (int rb = 0; rb < AE_RB; rb++) seen[rb] = 0.f;
#pragma unroll
  for (int rb = 0; rb < AE_RB; rb++) cls[rb] = row_class(j, rb);
#if !AE_DEEP
  if (any_tile && AE_J_LIVE) load_tile(j, 0);
#endif
#ifdef AE_HAS_KV_PREFETCH
  if (any_tile) {
#pragma unroll
    for (int rb = 0; rb < AE_RB; rb++) ae_prefetch_custom(cust[rb], j * AE_BN + 4 * hf, q0w + rb * 32, j * AE_BN, p);
  }
#endif
  // Drain every outstanding load (Q fragments, first tile) before the loop: with loads still
  // pending at the loop header the compiler's wait-count insertion makes the QK^T MFMAs of every
  // iteration wait for that iteration's K/V prefetch, which serialises the pipeline.
#if AE_DEEP
  __builtin_amdgcn_s_waitcnt(0xc07f);            // lgkmcnt(0); the Q rows and the first tile are waited for together
  request_next();
  request_next();
  wait_tile(j);
#else
  __builtin_amdgcn_s_waitcnt(0);
#endif
  __syncthreads();
#if AE_Q_VIA_LDS
#pragma unroll
  for (int rb = 0; rb < AE_RB; rb++)
#pragma unroll
    for (int ks = 0; ks < AE_D / 16; ks++)
      qf[rb][ks] = *(const __attribute__((address_space(3))) ae_elem8*)(
          qs + (rb * 32 + l32) * AE_KSTR + (ae_k_swz(2 * ks + hf, l32) << 4));
  __syncthreads();      // every wave has its fragments before the next request refills the rows' stages
#endif

#if AE_OWN_SOFTMAX
  static_assert(AE_RB == 1 && AE_WAVES_PER_EU >= 2, "one row block a wave, O in ordinary registers");
  float minus_ref = 0.f;       // the lane's row's reference, log2 units, negative
#endif
#if AE_FIRST_REST
  static_assert(AE_OWN_SOFTMAX, "weights up to 256");
  bool first = true;
#endif
  int stage = 0;
  while (AE_TRIPS_LEFT) {
#if AE_ROTATE
    const int jn = j + 1 == j_end ? j_first : j + 1;
#else
    const int jn = next_tile(j + AE_KW);
#endif
    int cls_n[AE_RB];
#pragma unroll
    for (int rb = 0; rb < AE_RB; rb++) cls_n[rb] = row_class(jn, rb);
#if AE_DEEP
    request_next();                              // into the stage that the last trip left
#else
    if (AE_HAS_NEXT) load_tile(jn, stage ^ 1);   // streams into the other stage while this one is used
#endif

    ae_lds_byte* ks_ = lds + stage * AE_STAGE_BYTES;
    ae_lds_byte* vs_ = ks_ + AE_K_BYTES;
    const int kv0 = j * AE_BN;
#if AE_WAVES_PER_EU == 1 && (AE_RB * (AE_NO + AE_NS) <= 256 || AE_O_SCALE_ONE)
    // (builds that use both register files: naming O as accumulator-file values once per tile keeps the
    // register allocator from moving parts of it between the files around the functor code.  Not where O
    // alone fills the accumulator file and the loop also rescales it: there the hint turns into spills -
    // measured 6.2 against 0.52 ms for the softmax at D 256, DV 512, while retention, whose normalisation
    // is deferred, gains from it: 1.00 -> 0.78 ms)
#pragma unroll
    for (int rb = 0; rb < AE_RB; rb++)
#pragma unroll
      for (int db = 0; db < AE_NDB; db++) asm volatile("" : "+a"(oacc[rb][db]));
#endif

#if AE_ANALYTIC && !defined(AE_HAS_KV_PREFETCH) && AE_WAVES_PER_EU >= 2
    // (wave uniform: some row of this wave sees a key of the tile.  Not where the functors also fetch custom inputs
    // tile by tile, which has to go on; not in the builds that fill the register file with one wave, which spill)
    bool active = kv0 <= q0w + AE_WROWS - 1 - AE_BAND_LO;
#if AE_BAND_HI != 0x7fffffff
    active = active && kv0 + AE_BN - 1 >= q0w - AE_BAND_HI;
#endif
    if (active && AE_J_LIVE)
#elif AE_KW > 1
    if (AE_J_LIVE)
#endif
    {
    // ---- S^T = K Q^T: every K fragment feeds one MFMA per row block -------------------------
    ae_f32x16 sacc[AE_RB][AE_NB];
#pragma unroll
    for (int rb = 0; rb < AE_RB; rb++)
#pragma unroll
      for (int nb = 0; nb < AE_NB; nb++)
#pragma unroll
        for (int r = 0; r < 16; r++) sacc[rb][nb][r] = 0.f;
    unsigned k_at = (unsigned)(unsigned long)ks_ + k_lane;
    asm("" : "+v"(k_at));                        // (a value of its own: not rebuilt per read from its parts)
    auto k_frag = [&](int f) AE_LAMBDA -> ae_elem8 {
      const int c = 2 * (f / AE_NB);
      return *(const __attribute__((address_space(3))) ae_elem8*)(
          (const ae_lds_byte*)(k_at ^ (unsigned)((c & (AE_KGRP - 1)) << 4)) + ((c & -AE_KGRP) << 4) + f % AE_NB * 32 * AE_KSTR);
    };
    constexpr int NKF = (AE_D / 16) * AE_NB;
    ae_elem8 kring[AE_K_AHEAD + 1];
    AE_SETPRIO(0);
#pragma unroll
    for (int f = 0; f < AE_K_AHEAD && f < NKF; f++) kring[f] = k_frag(f);
    AE_RING_FENCE();
#pragma unroll
    for (int f = 0; f < NKF; f++) {
      if (f + AE_K_AHEAD < NKF) kring[(f + AE_K_AHEAD) % (AE_K_AHEAD + 1)] = k_frag(f + AE_K_AHEAD);
#pragma unroll
      for (int rb = 0; rb < AE_RB; rb++)
        sacc[rb][f % AE_NB] = ae_mfma32(kring[f % (AE_K_AHEAD + 1)], qf[rb][f / AE_NB], sacc[rb][f % AE_NB]);
      AE_RING_FENCE();
    }

    AE_SETPRIO(1);
    unsigned v_at = (unsigned)(unsigned long)vs_ + v_lane;
    asm("" : "+v"(v_at));
    auto v_frag = [&](int f) AE_LAMBDA -> ae_elem8 {
      // slots 0..3 of k-step kk are kv rows rb0+4*hf+0..3, slots 4..7 rows rb0+8+4*hf+0..3
      // (rb0 and +8 are multiples of 8, so they do not change the swizzle)
      const int kk = f / AE_NDB;
      const int rb0 = (kk >> 1) * 32 + (kk & 1) * 16;
      const int pair = 2 * (f % AE_NDB);
      const ae_lds_byte* a0 = (const ae_lds_byte*)(v_at ^ (unsigned)((pair & AE_VSWM) << 5)) + ((pair & ~AE_VSWM) << 5) + rb0 * AE_VSTR;
      ae_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) ae_s16x4*)a0);
      ae_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) ae_s16x4*)(a0 + 8 * AE_VSTR));
      return __builtin_bit_cast(ae_elem8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    ae_elem8 pf[AE_RB][AE_BN / 16];
#pragma unroll
    for (int rb = 0; rb < AE_RB; rb++) {
      float s[AE_NS];
#pragma unroll
      for (int nb = 0; nb < AE_NB; nb++)
#pragma unroll
        for (int r = 0; r < 16; r++) s[nb * 16 + r] = sacc[rb][nb][r];
      const int kvb = kv0 + 4 * hf;
      ctx[rb].kv_base = kvb;

      // ---- mask (additive -inf before score_mod, attn_tl.py:124-137) --------------------------
#if !AE_ANALYTIC
      bool masked_here = false;    // some score of this row block was tested on this tile
#endif
#if AE_ANALYTIC
      const int qd = qrow[rb] - kvb;            // q - kv of score e is qd - ae_kv_off(e)
      if (kv0 + AE_BN - 1 > q0w + rb * 32 - AE_BAND_LO) {  // tile crosses the diagonal of this row block
#pragma unroll
        for (int e = 0; e < AE_NS; e++) s[e] = (qd >= ae_kv_off(e) + AE_BAND_LO) ? s[e] : AE_NEG_INF;
      }
#if AE_BAND_HI != 0x7fffffff
      if (kv0 < q0w + rb * 32 + 31 - AE_BAND_HI) {         // ... the far edge of the band
#pragma unroll
        for (int e = 0; e < AE_NS; e++) s[e] = (qd <= ae_kv_off(e) + AE_BAND_HI) ? s[e] : AE_NEG_INF;
      }
#endif
#elif AE_MASK_MODE == 2 && !(defined(AE_MASK_VALUE_ZERO) && AE_MASK_VALUE_ZERO)
      if (__builtin_amdgcn_ballot_w64(cls[rb] != 2) != 0) {   // some row of this block does not see the whole tile
        masked_here = true;
#pragma unroll
        for (int e = 0; e < AE_NS; e++) {
#if AE_HAS_MASK_MOD
          const bool vis = cls[rb] == 2 || (cls[rb] == 1 && ae_mask_mod(b, h, qrow[rb], kvb + ae_kv_off(e)));
#else
          const bool vis = cls[rb] != 0;
#endif
          s[e] = vis ? s[e] : AE_NEG_INF;
        }
      }
#elif AE_HAS_MASK_MOD
      {
        masked_here = true;
#pragma unroll
        for (int e = 0; e < AE_NS; e++)
          s[e] = ae_mask_mod(b, h, qrow[rb], kvb + ae_kv_off(e)) ? s[e] : AE_NEG_INF;
      }
#endif
#if AE_PAD_SCORES          // (not causal over equal lengths: behind the diagonal of every row)
      if (kv0 + AE_BN > p.seqlen_kv) {
#pragma unroll
        for (int e = 0; e < AE_NS; e++) s[e] = ae_kv_off(e) < p.seqlen_kv - kvb ? s[e] : AE_KV_PAD;
      }
#endif
#if AE_ANALYTIC
      {
        // the row's visible keys of this tile are an interval
        int lo_kv = kv0, hi_kv = kv0 + AE_BN - 1;
        hi_kv = hi_kv < p.seqlen_kv ? hi_kv : p.seqlen_kv - 1;
        hi_kv = hi_kv < qrow[rb] - AE_BAND_LO ? hi_kv : qrow[rb] - AE_BAND_LO;
#if AE_BAND_HI != 0x7fffffff
        lo_kv = lo_kv > qrow[rb] - AE_BAND_HI ? lo_kv : qrow[rb] - AE_BAND_HI;
#endif
        seen[rb] = lo_kv <= hi_kv ? 1.f : seen[rb];
      }
#else
      if (masked_here) {           // (an untested tile is visible to every row; a tile that the end of the sequence cuts holds a key)
        float top = s[0];
#pragma unroll
        for (int e = 1; e < AE_NS; e++) top = __builtin_fmaxf(top, s[e]);
        seen[rb] = top > AE_NEG_INF ? 1.f : seen[rb];
      } else {
        seen[rb] = 1.f;
      }
#endif

#if AE_OWN_SOFTMAX
      const float lane_top = ae_lane_max<AE_NS>(s);
      float over = __builtin_fmaf(lane_top, AE_SM_SCALE, -st[rb].AE_SM_M);
      if (__builtin_amdgcn_ballot_w64(over > AE_SM_TAU) != 0) {      // (the first tile; seldom later)
        over = ae_group_max(over);
        const float ref = over > AE_SM_TAU ? ae_group_max(lane_top) * AE_SM_SCALE : st[rb].AE_SM_M;
        const float o_scale = ae_exp(st[rb].AE_SM_M - ref);          // (1 for rows whose reference stays)
        minus_ref = -ref * AE_LOG2E;
        st[rb].AE_SM_M = ref;
        st[rb].AE_SM_R *= o_scale;
#pragma unroll
        for (int db = 0; db < AE_NDB; db++)
#pragma unroll
          for (int r = 0; r < 16; r++) oacc[rb][db][r] *= o_scale;
      }
#pragma unroll
      for (int e = 0; e < AE_NS; e++) s[e] = ae_exp2(__builtin_fmaf(s[e], AE_SM_SCALE * AE_LOG2E, minus_ref));
      st[rb].AE_SM_R += ae_lane_sum<AE_NS>(s);
      asm("" : "+v"(st[rb].AE_SM_R));          // (now: put off, the weights stay beside their fragments, 13 registers more)
#else
      // ---- user functors ----------------------------------------------------------------------
#if defined(AE_HAS_KV_PREFETCH) && AE_KV_COALESCED
      // per-score custom inputs: from the coalesced layout they were fetched in to the lanes that own them
      ae_stage_custom(cust[rb], lds + AE_KV_STAGES * AE_STAGE_BYTES + (wave * AE_RB + rb) * AE_KV_SCRATCH);
#endif
      ae_score_mod<AE_NS>(s, ctx[rb], cust[rb]);
      float o_scale = ae_online_fwd<AE_NS>(s, st[rb], ctx[rb], cust[rb]);
#endif
#ifdef AE_HAS_KV_PREFETCH
      // the functors are done with this tile's elements of the per-score custom inputs: request the next
      // tile's, which travel while the second product runs
      if (AE_HAS_NEXT) ae_prefetch_custom(cust[rb], jn * AE_BN + 4 * hf, q0w + rb * 32, jn * AE_BN, p);
#endif

#if AE_PAD_WEIGHTS
      if (kv0 + AE_BN > p.seqlen_kv) {
#pragma unroll
        for (int e = 0; e < AE_NS; e++) s[e] = ae_kv_off(e) < p.seqlen_kv - kvb ? s[e] : 0.f;
      }
#endif

      // ---- P -> B-operand fragments -----------------------------------------------------------
#pragma unroll
      for (int kk = 0; kk < AE_BN / 16; kk++)
#pragma unroll
        for (int t = 0; t < 8; t += 2) {
          typedef float ae_f32x2 __attribute__((ext_vector_type(2)));
          const ae_f32x2 x2 = {s[kk * 8 + t], s[kk * 8 + t + 1]};
          const ae_elem2 y2 = __builtin_convertvector(x2, ae_elem2);       // one packed conversion
          pf[rb][kk][t] = y2[0];
          pf[rb][kk][t + 1] = y2[1];
        }

#if AE_FIRST_REST
      if (first) {
        first = false;
#pragma unroll
        for (int kk = 0; kk < AE_BN / 16; kk++) {
          ae_elem8 rest;
#pragma unroll
          for (int t = 0; t < 8; t++) rest[t] = (ae_elem)(s[kk * 8 + t] - (float)pf[rb][kk][t]);
#pragma unroll
          for (int db = 0; db < AE_NDB; db++) oacc[rb][db] = ae_mfma32(v_frag(kk * AE_NDB + db), rest, oacc[rb][db]);
        }
      }
#endif

#if !AE_O_SCALE_ONE && !AE_OWN_SOFTMAX
      // skip the rescale when no row of this block changed its scale (wave-uniform branch)
      if (__builtin_amdgcn_ballot_w64(o_scale != 1.0f) != 0) {
#pragma unroll
        for (int db = 0; db < AE_NDB; db++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
#if AE_WAVES_PER_EU == 1
            // builds with one wave per SIMD keep O in the accumulator file: one register at a time through one
            // scratch register (as plain arithmetic the allocator wants all of O in ordinary registers)
            float o = oacc[rb][db][r], t;
            asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1"
                         : "+a"(o), "=&v"(t) : "v"(o_scale));
            oacc[rb][db][r] = o;
#else
            oacc[rb][db][r] *= o_scale;
#endif
          }
      }
#elif !AE_OWN_SOFTMAX
      (void)o_scale;
#endif
    }

    // ---- O^T += V^T P^T: every V fragment feeds one MFMA per row block ------------------------
    constexpr int NVF = (AE_BN / 16) * AE_NDB;
    ae_elem8 vring[AE_V_AHEAD + 1];
    AE_SETPRIO(2);
#pragma unroll
    for (int f = 0; f < AE_V_AHEAD && f < NVF; f++) vring[f] = v_frag(f);
    AE_RING_FENCE();
#pragma unroll
    for (int f = 0; f < NVF; f++) {
      if (f + AE_V_AHEAD < NVF) vring[(f + AE_V_AHEAD) % (AE_V_AHEAD + 1)] = v_frag(f + AE_V_AHEAD);
#pragma unroll
      for (int rb = 0; rb < AE_RB; rb++)
        oacc[rb][f % AE_NDB] = ae_mfma32(vring[f % (AE_V_AHEAD + 1)], pf[rb][f / AE_NDB], oacc[rb][f % AE_NDB]);
      AE_RING_FENCE();
    }
    }

    // the next tile must have landed before anyone reads it: direct loads are tracked by vmcnt
#if AE_DEEP
    wait_tile(j + AE_KW);
    __syncthreads();
    stage = stage == 2 ? 0 : stage + 1;
#else
    __builtin_amdgcn_s_waitcnt(0x0070 | 0x0f00 | 0x0000);  // vmcnt(0), expcnt/lgkmcnt untouched
    __syncthreads();
    stage ^= 1;
#endif
    j = jn;
#if AE_ROTATE
    left--;
#endif
#pragma unroll
    for (int rb = 0; rb < AE_RB; rb++) cls[rb] = cls_n[rb];
  }

  // ---- epilogue -------------------------------------------------------------------------------
#if AE_OWN_SOFTMAX
  st[0].AE_SM_R = ae_group_sum(st[0].AE_SM_R);
#endif
#if AE_KW > 1
  // Every wave leaves its O and its row state in LDS (the stages are free: the loop ended with a barrier; element e of
  // lane l at 16 * ((e / 4) * 64 + l) + 4 * (e % 4), so that all accesses are 16 bytes a lane in lane order), then takes
  // the elements [kg * AE_NE, (kg + 1) * AE_NE) of its rows over all groups.
  {
    constexpr int AE_NE = AE_NO / AE_KW;
    typedef __attribute__((address_space(3))) ae_f32x4 lds_f4;
    typedef __attribute__((address_space(3))) float lds_f;
    ae_lds_byte* xo = (ae_lds_byte*)ae_smem;                                  // [wave][AE_NO * 64] floats
    lds_f* xs = (lds_f*)(xo + AE_KW * AE_NWAVES * AE_NO * 256);               // [wave][m, r, seen][64]
#pragma unroll
    for (int e = 0; e < AE_NO; e += 4) {
      const ae_f32x16& a = oacc[0][e >> 4];
      *(lds_f4*)(xo + wave_wg * (AE_NO * 256) + (e >> 2) * 1024 + lane * 16) =
          (ae_f32x4){a[e & 15], a[(e & 15) + 1], a[(e & 15) + 2], a[(e & 15) + 3]};
    }
#if AE_KW_SOFTMAX
    xs[(wave_wg * 3 + 0) * 64 + lane] = st[0].AE_SM_M;
    xs[(wave_wg * 3 + 1) * 64 + lane] = st[0].AE_SM_R;
#endif
    xs[(wave_wg * 3 + 2) * 64 + lane] = seen[0];
    __syncthreads();
    float w[AE_KW];
    // a group that met a visible key of the row counts, whatever its weight is: one whose visible scores are all NaN
    // keeps the reference it started with (weight 0) and its NaN has to reach the row all the same
    bool live[AE_KW];
    bool row_seen = false;
#if AE_KW_SOFTMAX
    float mg[AE_KW], top = AE_NEG_INF, r_sum = 0.f;
#endif
#pragma unroll
    for (int k = 0; k < AE_KW; k++) {
      const int wk = (k * AE_NWAVES + wave) * 3;
      live[k] = ae_group_max(xs[(wk + 2) * 64 + lane]) > 0.f;
      row_seen = row_seen || live[k];
      w[k] = 1.f;
#if !AE_KW_SOFTMAX
      live[k] = true;      // (no row state: what a group's tiles gave is the row's, the weights of masked keys included)
#else
      mg[k] = xs[wk * 64 + lane];
      top = live[k] ? __builtin_fmaxf(top, mg[k]) : top;
#endif
    }
#if AE_KW_SOFTMAX
#pragma unroll
    for (int k = 0; k < AE_KW; k++) {
      w[k] = ae_exp(mg[k] - top);
      r_sum += live[k] ? xs[((k * AE_NWAVES + wave) * 3 + 1) * 64 + lane] * w[k] : 0.f;
    }
    st[0].AE_SM_M = top;
    st[0].AE_SM_R = r_sum;
#endif
    float o[AE_NE];
#pragma unroll
    for (int e = 0; e < AE_NE; e++) o[e] = 0.f;
#pragma unroll
    for (int k = 0; k < AE_KW; k++)
#pragma unroll
      for (int e = 0; e < AE_NE; e += 4) {
        const ae_f32x4 v = *(const lds_f4*)(xo + (k * AE_NWAVES + wave) * (AE_NO * 256) + ((kg * AE_NE + e) >> 2) * 1024 + lane * 16);
#pragma unroll
        for (int t = 0; t < 4; t++) o[e + t] += live[k] ? v[t] * w[k] : 0.f;
      }
    float frs[AE_N_ROWSCALES > 0 ? AE_N_ROWSCALES : 1];
    frs[0] = 0.f;
    if (any_tile && row_seen) {
      ae_epilogue<AE_NE>(o, st[0], frs, ctx[0], cust[0]);
    } else {
#pragma unroll
      for (int e = 0; e < AE_NE; e++) o[e] = 0.f;
#pragma unroll
      for (int i = 0; i < AE_N_ROWSCALES; i++) frs[i] = AE_NEG_INF;
    }
#if AE_MERGE_LAST
    const int64_t first = (((int64_t)b * p.seqlen_q + q0) * p.heads_q + h) * n_split;
    const int rows_here = p.seqlen_q - q0 < AE_BM ? p.seqlen_q - q0 : AE_BM;
    const int row_step = p.heads_q * n_split;
    __amdgpu_buffer_rsrc_t part = __builtin_amdgcn_make_buffer_rsrc(
        p.partial_o + first * AE_DV, 0, ((rows_here - 1) * row_step + n_split) * (AE_DV * 4), 0x00020000);
    const bool merged = p.tail_slots != 0;
#endif
    if (q_ok[0]) {
#if AE_MERGE_LAST
      const int at = (qrow[0] - q0) * row_step + split;
#endif
#if AE_NSPLIT > 1
      const int64_t prow = ((((int64_t)b * p.seqlen_q + qrow[0]) * p.heads_q + h) * n_split) + split;
      float* po = p.partial_o + prow * AE_DV;
#else
      ae_elem* po = (ae_elem*)p.out + (int64_t)b * p.o_stride_b + (int64_t)qrow[0] * p.o_stride_s + (int64_t)h * p.o_stride_h;
#endif
#pragma unroll
      for (int e = 0; e < AE_NE; e += 4) {
        const int ea = kg * AE_NE + e;                      // element ea .. ea + 3: four neighbouring columns
        const int col = (ea >> 4) * 32 + ((ea & 15) >> 2) * 8 + hf * 4;
#if AE_MERGE_LAST
        if (merged)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(ae_u32x4, (ae_f32x4){o[e], o[e + 1], o[e + 2], o[e + 3]}), part,
                                                 (at * AE_DV + col) * 4, 0, kAeDeviceScope);
        else
#endif
#if AE_NSPLIT > 1
        *(ae_f32x4*)(po + col) = (ae_f32x4){o[e], o[e + 1], o[e + 2], o[e + 3]};
#else
        *(ae_elem4*)(po + col) = (ae_elem4){(ae_elem)o[e], (ae_elem)o[e + 1], (ae_elem)o[e + 2], (ae_elem)o[e + 3]};
#endif
      }
      if (hf == 0 && kg == 0) {
#pragma unroll
        for (int i = 0; i < AE_N_ROWSCALES; i++)
#if AE_MERGE_LAST
          if (merged) __hip_atomic_store(p.partial_rs + first + at, frs[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          else
#endif
#if AE_NSPLIT > 1
          p.partial_rs[(int64_t)i * p.batch * p.seqlen_q * p.heads_q * n_split + prow] = frs[i];
#else
          p.rowscale_out[i][((int64_t)b * p.heads_q + h) * p.seqlen_q + qrow[0]] = frs[i];
#endif
      }
    }
#if AE_MERGE_LAST
    if (!merged) return;
    int* const counter = (int*)(p.partial_rs + (int64_t)p.batch * p.seqlen_q * p.heads_q * n_split) + (int64_t)bh * n_qt + qt;
    if (!ae_count_in(counter, n_split, tid == 0, (__attribute__((address_space(3))) int*)xs)) return;
    ae_merge_rows<AE_NT>(p, first, row_step, tid, rows_here, n_split, [&](int r, int col, ae_f32x4 acc, float merged) AE_LAMBDA {
      ae_elem4 w;
#pragma unroll
      for (int c = 0; c < 4; c++) w[c] = (ae_elem)acc[c];
      *(ae_elem4*)((ae_elem*)p.out + (int64_t)b * p.o_stride_b + (int64_t)(q0 + r) * p.o_stride_s + (int64_t)h * p.o_stride_h + col) = w;
      if (col == 0) p.rowscale_out[0][((int64_t)b * p.heads_q + h) * p.seqlen_q + q0 + r] = merged;
    });
#endif
  }
#elif AE_NO > 128 && AE_NSPLIT == 1
  // wide value heads: the epilogue functor (elementwise over the value columns) runs one 32-column block at a
  // time; a copy of all of O next to its accumulators would not fit the register file
#pragma unroll
  for (int rb = 0; rb < AE_RB; rb++) {
    float frs[AE_N_ROWSCALES > 0 ? AE_N_ROWSCALES : 1];
    frs[0] = 0.f;
    const bool row_seen = ae_group_max(seen[rb]) > 0.f;     // (both lanes of a row, or neither)
    ae_elem* optr = (ae_elem*)p.out + (int64_t)b * p.o_stride_b + (int64_t)qrow[rb] * p.o_stride_s +
                    (int64_t)h * p.o_stride_h;
#pragma unroll
    for (int db = 0; db < AE_NDB; db++) {
      // (read where it is used: as plain copies the accumulator reads of EVERY block move to the front, which
      // takes the whole register file and spills; a volatile asm statement stays behind the previous block's stores)
      float o[16];
#pragma unroll
      for (int r = 0; r < 16; r++) asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(o[r]) : "a"(oacc[rb][db][r]));
      if (any_tile && row_seen) {
        ae_epilogue<16>(o, st[rb], frs, ctx[rb], cust[rb]);
      } else {
#pragma unroll
        for (int r = 0; r < 16; r++) o[r] = 0.f;
#pragma unroll
        for (int i = 0; i < AE_N_ROWSCALES; i++) frs[i] = AE_NEG_INF;
      }
      if (q_ok[rb]) {
#pragma unroll
        for (int rg = 0; rg < 4; rg++) {
          ae_elem4 w;
#pragma unroll
          for (int t = 0; t < 4; t++) w[t] = (ae_elem)o[rg * 4 + t];
          *(ae_elem4*)(optr + db * 32 + rg * 8 + hf * 4) = w;
        }
      }
    }
    if (q_ok[rb] && hf == 0) {
#pragma unroll
      for (int i = 0; i < AE_N_ROWSCALES; i++)
        p.rowscale_out[i][((int64_t)b * p.heads_q + h) * p.seqlen_q + qrow[rb]] = frs[i];
    }
  }
#else
#pragma unroll
  for (int rb = 0; rb < AE_RB; rb++) {
    float o[AE_NO];
#pragma unroll
    for (int db = 0; db < AE_NDB; db++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[db * 16 + r] = oacc[rb][db][r];
    float frs[AE_N_ROWSCALES > 0 ? AE_N_ROWSCALES : 1];
    frs[0] = 0.f;
    const bool row_seen = ae_group_max(seen[rb]) > 0.f;     // (both lanes of a row, or neither)
    // no visible kv block for this q-tile, or no visible key for this row: out = 0 (blockattn_tl.py:153-160),
    // rowscales = -inf.  (selected after the functor and, where they are converted, on the converted pairs: as the two
    // sides of a branch every element was a register to clear and a conversion of its own)
    const bool live = any_tile && row_seen;
    ae_epilogue<AE_NO>(o, st[rb], frs, ctx[rb], cust[rb]);
#pragma unroll
    for (int i = 0; i < AE_N_ROWSCALES; i++) frs[i] = live ? frs[i] : AE_NEG_INF;
    auto out4 = [&](int e) AE_LAMBDA -> ae_elem4 {
      typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
      const u32x2 w = __builtin_bit_cast(u32x2, (ae_elem4){(ae_elem)o[e], (ae_elem)o[e + 1], (ae_elem)o[e + 2], (ae_elem)o[e + 3]});
      return __builtin_bit_cast(ae_elem4, (u32x2){live ? w[0] : 0u, live ? w[1] : 0u});
    };
#if AE_NSPLIT > 1
    // partial result of this split: fp32, rows ordered (batch, q position, head) so that the merge
    // kernel sees them as B x (Sq*Hq) "heads" of a one-token decode and writes out [B,Sq,Hq,DV].  O leaves through the
    // wave's share of the tile ring, a row's columns as one contiguous piece: straight from the accumulators a
    // store instruction writes 16 bytes of each of 64 rows, lines that the L2 has to put together out of eight pieces.  Up
    // to 12 MB of them go past the caches, which have less to write back when the launch ends; more of them wait for
    // memory beside the cache's reads.  B5 H8 Sq77 Skv842 D128 (8 MB): the call 16.9 us, 17.3 through the caches, 15.0 past
    // them; B1 H32 Sq128 Skv8192 (17 MB): 42.7, 42.2, 43.4.
    {
      constexpr int REGION = 2 * AE_STAGE_BYTES / AE_NWAVES;                            // bytes of LDS a wave may use
      constexpr int NP = 32 * AE_DV * 4 <= REGION ? 1 : (16 * AE_DV * 4 <= REGION ? 2 : 4);   // passes over the columns
      constexpr int CPR = AE_DV / 4 / NP;                                               // 16-byte chunks of a row and pass
      constexpr int SW = (CPR & -CPR) < 32 ? (CPR & -CPR) - 1 : 31;
      static_assert(AE_RB == 1 && 32 * CPR * 16 <= REGION && AE_NDB % NP == 0 && 32 * CPR % 64 == 0, "the rows fit the wave's share of the tile ring");
      typedef __attribute__((address_space(3))) ae_f32x4 lds_f4;
      int le = lane;
      asm volatile("" : "+v"(le));
      ae_lds_byte* os = lds + wave * REGION;
      const int64_t row0 = ((int64_t)b * p.seqlen_q + q0w) * p.heads_q + h;
      const bool past = (int64_t)p.batch * p.seqlen_q * p.heads_q * (n_split * AE_DV * 4) <= 12 << 20;
#pragma unroll
      for (int ps = 0; ps < NP; ps++) {
        ae_lds_byte* orow = os + (le & 31) * (CPR * 16);
#pragma unroll
        for (int db = 0; db < AE_NDB / NP; db++)
#pragma unroll
          for (int rg = 0; rg < 4; rg++) {
            ae_f32x4 w;
#pragma unroll
            for (int t = 0; t < 4; t++) w[t] = live ? o[(ps * (AE_NDB / NP) + db) * 16 + rg * 4 + t] : 0.f;
            *(lds_f4*)(orow + (((db * 8 + rg * 2 + (le >> 5)) ^ (le & SW)) << 4)) = w;
          }
        // (the rows were written by other lanes of this wave: LDS instructions of a wave complete in order)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        auto leave = [&](auto past_tag) AE_LAMBDA {
#pragma unroll 8
          for (int i = 0; i < 32 * CPR / 64; i++) {
            const int row = (i * 64 + le) / CPR, c = (i * 64 + le) % CPR;
            const ae_f32x4 w = *(const lds_f4*)(os + row * (CPR * 16) + ((c ^ (row & SW)) << 4));
            ae_f32x4* at = (ae_f32x4*)(p.partial_o + ((row0 + (int64_t)row * p.heads_q) * n_split + split) * AE_DV + (ps * CPR + c) * 4);
            if (AE_EVEN_Q || q0w + row < p.seqlen_q) {
              if (decltype(past_tag)::value) __builtin_nontemporal_store(w, at);
              else *at = w;
            }
          }
        };
        if (past) {
          asm volatile("" ::: "memory");                 // (else the two loops become one, of plain stores)
          leave(ae_const_bool<true>());
        } else {
          leave(ae_const_bool<false>());
        }
      }
    }
    if (q_ok[rb] && hf == 0) {
      const int64_t prow = ((((int64_t)b * p.seqlen_q + qrow[rb]) * p.heads_q + h) * n_split) + split;
#pragma unroll
      for (int i = 0; i < AE_N_ROWSCALES; i++)
        p.partial_rs[(int64_t)i * p.batch * p.seqlen_q * p.heads_q * n_split + prow] = frs[i];
    }
#elif AE_O_VIA_LDS
    {
      // (addresses from a copy of the lane id that the compiler cannot trace back to the prologue's, which have
      // the same form: it would keep those in registers across the loop)
      int le = lane;
      asm volatile("" : "+v"(le));
      ae_lds_byte* orow = lds + wave * (AE_WROWS * AE_VSTR) + (rb * 32 + (le & 31)) * AE_VSTR + (le >> 5) * 8;
      const int osw = le & (AE_VCPR - 1);
#pragma unroll
      for (int db = 0; db < AE_NDB; db++)
#pragma unroll
        for (int rg = 0; rg < 4; rg++) {
          *(__attribute__((address_space(3))) ae_elem4*)(orow + (((db * 4 + rg) ^ osw) << 4)) = out4(db * 16 + rg * 4);
        }
    }
    if (q_ok[rb] && hf == 0) {
#pragma unroll
      for (int i = 0; i < AE_N_ROWSCALES; i++)
        p.rowscale_out[i][((int64_t)b * p.heads_q + h) * p.seqlen_q + qrow[rb]] = frs[i];
    }
#else
    if (q_ok[rb]) {
      ae_elem* optr = (ae_elem*)p.out + (int64_t)b * p.o_stride_b + (int64_t)qrow[rb] * p.o_stride_s +
                      (int64_t)h * p.o_stride_h;
#pragma unroll
      for (int db = 0; db < AE_NDB; db++)
#pragma unroll
        for (int rg = 0; rg < 4; rg++) {
          *(ae_elem4*)(optr + db * 32 + rg * 8 + hf * 4) = out4(db * 16 + rg * 4);
        }
      if (hf == 0) {
#pragma unroll
        for (int i = 0; i < AE_N_ROWSCALES; i++)
          p.rowscale_out[i][((int64_t)b * p.heads_q + h) * p.seqlen_q + qrow[rb]] = frs[i];
      }
    }
#endif
  }
#if AE_O_VIA_LDS
  // (the rows were written by other lanes of this wave: LDS instructions of a wave complete in order)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  {
    ae_elem* og = (ae_elem*)p.out + (int64_t)b * p.o_stride_b + (int64_t)h * p.o_stride_h;
    const ae_lds_byte* os = lds + wave * (AE_WROWS * AE_VSTR);
    int le = lane;
    asm volatile("" : "+v"(le));
#pragma unroll
    for (int i = 0; i < AE_O_LOADS; i++) {
      const int n = i * 64 + le;
      const int row = n / AE_VCPR;
      const int c = n % AE_VCPR;
      const ae_elem8 w = *(const __attribute__((address_space(3))) ae_elem8*)(
          os + row * AE_VSTR + ((c ^ (row & (AE_VCPR - 1))) << 4));
      if (AE_EVEN_Q || q0w + row < p.seqlen_q) *(ae_elem8*)(og + (int64_t)(q0w + row) * p.o_stride_s + c * 8) = w;
    }
  }
#endif
#endif  // wide value heads
}

#ifdef AE_COMBINE_THREADS       // (a caller that wants both kernels in one module)
#include "ae_combine.h"
#endif
