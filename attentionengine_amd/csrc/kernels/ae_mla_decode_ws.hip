// MLA (shared latent KV) split-KV decode for gfx950 / CDNA4, wave-specialised: online softmax only.
//
// Same role as ae_mla_decode.hip (the reference's TileLang MLA decode template,
// attention_engine/core/template/tl_template/attn/mla_decode_tl.py: flash_attn_split 104-179, and the
// CuTe/FlashMLA split kernel, core/template/cute_template_kvshared/kernels/splitkv_mla.cu:1061-1393),
// for the case the lowering has proven to be the online softmax of `score * constant`
// (attn_script/mha.py:47-72); anything else uses ae_mla_decode.hip, which runs the generated functors.
//
// Why a second kernel: in ae_mla_decode.hip every one of 8 waves reads the whole KV tile from LDS for
// both products (416 KiB of LDS reads per 32-token tile and workgroup) and the two value halves of a
// head block compute the same scores; LDS bandwidth bounds it at ~0.21 ms for B128 H128 S4096.  Here
// the waves of a workgroup (64 query heads of one (batch, kv head, split)) have different jobs:
//   * 2 "score waves" (32 heads each): S^T[kv,head] = K Q^T with v_mfma_f32_32x32x16 (Q^T in registers for
//     the whole kernel, K fragments from LDS, each feeding a 32x32 block: with 16 heads per wave the four
//     waves' fragment reads, 144 KiB per tile, took 2.6x the time of their MFMAs), lazy online softmax,
//     P^T written to LDS as the B operand of the second product, per-head rescale factors next to it;
//   * 4 "value waves" (a quarter of the value columns each, all 64 heads): O^T[dv,head] += V^T P^T with
//     v_mfma_f32_16x16x32, paged 32x32x16 (AE_VB), V^T fragments read from the SAME LDS rows through ds_read_b64_tr_b16,
//     every fragment feeding all blocks of heads.
// Wave i runs on SIMD i % 4.  The workgroup is launched with 8 waves: waves 0, 1 are the score waves
// (SIMD 0, 1: 1152 matrix-pipe cycles per tile each), waves 2, 3, 6, 7 the value waves (two each on SIMD
// 2, 3: 2 x 512 cycles), waves 4, 5 leave at once (AE_HPW 16, paged cache: they request the tiles, AE_LOADER_WAVES) - so the four SIMDs carry about the same MFMA work.
// The score waves run one tile ahead of the value waves: one workgroup barrier per tile hands P over.
// Scores are computed once: 124 KiB of LDS reads per tile instead of 416.  KV tiles go HBM -> LDS
// directly (16 B per lane, chunk-swizzled as in ae_mla_decode.hip), AE_NSTAGE tiles deep; a trip ends by
// waiting until only the newest tile request is outstanding.
//
// AE_HPW (heads per workgroup): 64 is the form above.  32 and 16 are for launches that 64-head workgroups spread thin -
// few query heads, or so few sequences that the kv axis is split over many workgroups and every one of them pays for the
// fp32 partial results of 64 heads.  A trip of the 64-head form is one score wave's instruction stream (36 MFMAs, 36
// fragment reads, the softmax of 16 scores a lane: 0.81 us in split launches of a small batch, 1.1 where every CU is busy
// and the clock at the power cap); here 16 heads and 16 of the tile's 32 keys make up a score
// wave's share (v_mfma_f32_16x16x32: 18 MFMAs, 18 reads, 4 scores a lane), two waves per 16 heads, which exchange their
// maxima through LDS at the end of a trip and so keep one reference.  The value waves have 128 columns x 16 or 32 heads.  Per head the tile is fetched and read two or four times as often as with 64 heads, which is why the
// large launches keep that form.
//
// Configuration ("ae_config.h"): AE_HPW AE_D1 AE_D2 AE_DV AE_DTYPE_BF16 AE_N_ROWSCALES AE_NSPLIT (1: the kv axis is not split
// and the kernel writes out; more: p.num_splits says how often, ae_combine.hip merges) AE_PAGED (1: the cache is paged, rows are found through ae_attn_params.block_table and
// every batch entry has its own length seqlens_k[b], as in the reference's
// cute_template_kvshared/kernels/params.h:33-36; a kv tile never straddles two pages), plus AE_SM_SCALE (the constant c > 0) and AE_SM_M / AE_SM_R (names of the
// running-max and running-sum fields of ae_rowstate).  Functors used ("ae_functors.h"): ae_rowstate,
// ae_rowstate_init, ae_epilogue, ae_load_custom.

#define AE_LAYOUT 1
#include "ae_hip.h"
#include "ae_config.h"
#include "ae_device.h"
#include "ae_functors.h"

#ifndef AE_PAGED
#define AE_PAGED 0
#endif
// 0 (paged cache): never asked to split the entries by their lengths (ae_tile_cfg.paged 1).  Asked at run time, a launch of equal
// spans waits for the answer in front of its first request, 64 heads a workgroup: B33 H128 up to 3968 tokens 52.8 us, 52.0 with 0, B56
// 5056 81.0 and 80.4.
#ifndef AE_BY_LENGTH
#define AE_BY_LENGTH 1
#endif
#define AE_D (AE_D1 + AE_D2)
#define AE_NWAVES 8
#define AE_NT (AE_NWAVES * 64)
#ifndef AE_HPW
#define AE_HPW 64
#endif
#define AE_HEADS_PER_WG AE_HPW
#define AE_NSB (AE_HPW == 64 ? 2 : AE_HPW / 16)      // head blocks of the score waves: of 32 heads, or of 16
// Heads of a value wave's block, and columns of its V^T fragments: 16 (v_mfma_f32_16x16x32) or 32 (32x32x16).  16x16x32 takes the
// same matrix-pipe cycles and a sixth less power a product, twice the instructions.  The dense launch of 64 heads a workgroup is at the
// socket's power cap and its value waves have the issue slots: 32 -> 16, us, B128 H128 Skv4096 bf16 171.4 -> 166.8, fp16 184.3 ->
// 177.5, B64 Skv2000 fp16 58.6 -> 57.6, split B24 Skv4000 bf16 45.8 -> 45.0, B16 H64 Skv8000 42.7 either way.  A paged batch whose
// entries have different lengths leaves CUs idle and the clock up, and there the instructions count: B23 H128 up to 6848 tokens
// 52.4 -> 53.6, B56 5056 80.6 -> 82.1, B44 H64 2944 33.7 -> 34.4.  (The score waves' instruction stream is the trip: 32x32x16.)
#define AE_VB (AE_HPW == 64 && AE_PAGED ? 32 : 16)
#define AE_NHB (AE_HPW / AE_VB)           // head blocks of a value wave
#define AE_BN 32                          // kv rows per tile
#if AE_HPW == 64
#define AE_NKS (AE_D / 16)                // 16-deep k-steps of S^T = K Q^T
#else
#define AE_NKS (AE_D / 32)                // 32-deep ones
#endif
// 1: the tiles are requested by two waves of their own - waves 4 and 5, which 16 heads a workgroup leave idle - on the score
// waves' SIMDs.  A trip of 16 heads is bound by the serial chain of each wave (the LDS pipe busy for 830 of its 1500 cycles):
// a value wave that first issues nine requests, 16 cycles each, comes late to its products.  Paged cache, 128 heads, one
// split: 0.647 -> 0.533 us a trip, 0.9 us more until the first; B8 H128, 2048 tokens at most 19.8 -> 18.4 us, B6 H64 5568
// 21.5 -> 19.9, splits of two to four tiles the same.  Not for the dense cache: its requests take two VALU instructions
// each to step an address, which there delay the score waves (0.600 -> 0.606; four request waves of three a SIMD 0.592
// and, paged, 0.568).  Nor with 32 heads, where the score waves are waves 4 and 5 too (four more waves: 0.81 -> 0.87).
#define AE_LOADER_WAVES (AE_HPW == 16 && AE_PAGED)
#define AE_NLOADERS (AE_LOADER_WAVES ? 2 : 4)      // else the value waves also request the KV tiles
#define AE_DVW (AE_DV / 4)                // value columns of one value wave
#define AE_NDB (AE_DVW / AE_VB)           // dv blocks of a value wave
#define AE_NO (AE_DVW * AE_VB / 64)       // output elements per lane and head block
#define AE_KSTR (AE_D * 2)                // LDS row pitch, bytes (unpadded: swizzled)
#define AE_STAGE_BYTES (AE_BN * AE_KSTR)
#define AE_CPR (AE_D / 8)                 // 16-byte chunks per K row
#define AE_CPR1 (AE_D1 / 8)
#define AE_BLOCKS ((AE_BN * AE_CPR) / 64) // 1 KiB blocks per tile
#define AE_LOADS ((AE_BLOCKS + AE_NLOADERS - 1) / AE_NLOADERS)
#define AE_BURSTS (AE_LOADS <= 16 ? 2 : 3)   // a wave's loads of one tile go out as two or three bursts, burst i from load AE_LB(i)
#define AE_LB(i) (((i) * AE_LOADS + AE_BURSTS - 1) / AE_BURSTS)
#ifndef AE_NSTAGE
#define AE_NSTAGE 4
#endif
#define AE_PTAB 1024                      // paged cache: block-table entries of one split kept in LDS
#define AE_WHOLE_TABLE 512                // ... or of the whole table, up to this
#define AE_PSTR 80                        // LDS pitch of one head's P row (32 kv * 2 B, padded against bank conflicts)
#define AE_P_BYTES (AE_HEADS_PER_WG * AE_PSTR)
#define AE_X_BYTES (AE_HEADS_PER_WG * 4 + 16)   // per-head rescale factors + one flag word per head block
#define AE_XMAX_BYTES (AE_HPW == 64 ? 0 : AE_HPW * 8)   // the row maxima of a tile's two halves
#define AE_FIN (AE_HPW == 64 ? 2 : 3)                   // final row state per head: m, r (of each half)
#define AE_TAU2 8.0f                      // the running maximum (log2 units) is refreshed only when it moved by more
#define AE_SWZ(r) ((((r) >> 1) & 3) * 2 + (((r) >> 3) & 1))
#define AE_VMCNT(n) (0x0F70 | ((n) & 15) | (((n) >> 4) << 14))
#define AE_VMCNT_LGKM0(n) (0x0070 | ((n) & 15) | (((n) >> 4) << 14))
#ifndef AE_AHEAD
#define AE_AHEAD (AE_HPW == 64 ? 4 : 6)
#endif
#define AE_RING (AE_AHEAD + 1)

static_assert(AE_D1 % 32 == 0 && AE_D2 % 32 == 0, "latent / rope dims must be multiples of 32");
static_assert(AE_HPW == 64 || AE_HPW == 32 || AE_HPW == 16, "two blocks of 32 heads, or one or two of 16");
static_assert(AE_D % 64 == 0, "two accumulation chains over the k-steps");
static_assert(AE_DV % 128 == 0 && AE_DV <= AE_D1, "V must be a prefix of the latent part, four 32-column blocks wide");
static_assert(AE_CPR % 8 == 0 && AE_CPR1 % 8 == 0, "chunk groups of eight must not straddle the two K tensors");
static_assert((AE_BN * AE_CPR) % 64 == 0, "tile must be a whole number of 1 KiB blocks");
static_assert(AE_LB(1) <= 8 && AE_LOADS >= AE_BURSTS && AE_BLOCKS >= AE_LOADS, "bursts of at most eight loads per wave and tile");
static_assert(2 * AE_LOADS <= 63 && AE_NSTAGE == 4, "the wait counter holds the requests in flight");
// chunk exchange of the results in LDS: inside groups that divide a head's chunks (16 where there are as many)
#define AE_OSW1 ((AE_DVW / 8) & -(AE_DVW / 8))
#define AE_OSW (AE_OSW1 < 16 ? AE_OSW1 - 1 : 15)
static_assert(AE_DV * AE_HEADS_PER_WG * 4 <= AE_NSTAGE * AE_STAGE_BYTES, "the results of 64 heads fit the tile stages");
static_assert(AE_DVW % 64 == 0, "a value wave's first chunk is a multiple of eight, a block of heads leaves in whole instructions");
static_assert(AE_NSTAGE >= 3, "a tile is multiplied by K one trip before it is multiplied as V");

// 1 (single-split builds only, a measurement switch): every workgroup reports the shader-clock cycles (s_memtime)
// and the constant-rate 100 MHz ticks (s_memrealtime) between its entry and its last store, as two 64-bit values
// at ((unsigned long long*)p.partial_o)[2 * blockIdx.x] - a buffer a single-split launch does not otherwise use -
// and, behind the pairs of all workgroups (at index 2 * gridDim.x + 4 * blockIdx.x), four more tick values of one
// value wave: entry, first tile landed, last trip done, last store acknowledged (absolute 100 MHz ticks).
#ifndef AE_CLOCK_STAMPS
#define AE_CLOCK_STAMPS 0
#endif
static_assert(!AE_CLOCK_STAMPS || AE_NSPLIT == 1, "the clock stamps go where a split launch keeps its partial results");
#if AE_PAGED
#include "ae_mla_paged.h"
#endif

typedef __attribute__((address_space(3))) unsigned char ae_lds_byte;
typedef __attribute__((address_space(3))) float ae_lds_f32;
typedef __attribute__((address_space(3))) int ae_lds_i32;
template <bool B> struct ae_const_bool { static constexpr bool value = B; };
template <int I> struct ae_const_int { static constexpr int value = I; };

extern "C" __global__ __launch_bounds__(AE_NT) __attribute__((amdgpu_waves_per_eu(2, 2)))
void ae_mla_decode_split_kernel(const ae_attn_params p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char ae_smem[];
  ae_lds_byte* lds = (ae_lds_byte*)ae_smem;                     // AE_NSTAGE kv tiles
  ae_lds_byte* pbuf = lds + AE_NSTAGE * AE_STAGE_BYTES;         // 2 x P^T [head][kv]
  ae_lds_byte* xbuf = pbuf + 2 * AE_P_BYTES;                    // 2 x (rescale factors, flags)
  ae_lds_f32* xmax = (ae_lds_f32*)(xbuf + 2 * AE_X_BYTES);      // 2 x row maxima [half][head]
  ae_lds_f32* fin = xmax + 2 * (AE_XMAX_BYTES / 4);             // final (m, r) per head
#if AE_PAGED
  ae_lds_i32* ptab = (ae_lds_i32*)(fin + AE_FIN * AE_HEADS_PER_WG);  // AE_PTAB page numbers: this split's part of the block table
#endif

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool score_wave = wave < 2 || (AE_HPW == 32 && (wave == 4 || wave == 5));
  const bool requests = AE_LOADER_WAVES ? wave == 4 || wave == 5 : !score_wave;      // (waves that request the tiles)
#if AE_CLOCK_STAMPS
  const unsigned long long ae_t0 = __builtin_amdgcn_s_memtime();
  const unsigned long long ae_w0 = __builtin_amdgcn_s_memrealtime();
#endif

  // ---- which (head tile, split, kv head, batch): 1-D grid, ids 8 apart share their KV range ---------
  // (What a workgroup does before its first tile is requested is a serial chain that a short launch pays in full: the
  // integer divisions are left out where a shift does - one latent head, a power of two of head tiles, of tokens a page.
  // The number of splits is the launch's: one build serves every count above one, and writes where the host planned.)
  int group = p.heads_q;
  if (__builtin_expect(p.heads_kv != 1, 0)) group /= p.heads_kv;
  const int n_ht = (int)((unsigned)(group + AE_HEADS_PER_WG - 1) / AE_HEADS_PER_WG);
  const int wg = blockIdx.x;
  int ht, u8;
  if (__builtin_expect((n_ht & (n_ht - 1)) != 0, 0)) {
    ht = (wg >> 3) % n_ht;
    u8 = (wg >> 3) / n_ht;
  } else {
    ht = (wg >> 3) & (n_ht - 1);
    u8 = (wg >> 3) >> __builtin_ctz(n_ht);
  }
  const unsigned u = (unsigned)(u8 * 8 + (wg & 7));      // flattened (batch, kv head, split)
#if AE_NSPLIT == 1
  const int n_split = 1, per_split = p.kv_per_split;
  int split = 0, b = u, hk = 0;
#if AE_PAGED
  constexpr bool by_length = false;
  constexpr int len_b = 0;
  constexpr bool whole_table = false;
#endif
#else
  const int n_split = p.num_splits;
  int units = n_split, split, hk = 0;
#if AE_PAGED
  if (ae_mla_odd_units(p, n_ht)) units |= 1;
#endif
  int b;
#if AE_PAGED
  // (splits by the entries' lengths: see ae_split_by_length)
#if AE_BY_LENGTH
  const bool by_length = p.tail_slots != 0;
#else
  constexpr bool by_length = false;
#endif
  // (rows may lie any distance apart: 64 bits, as for `pages` below)
  const int64_t all_ints = (int64_t)(p.batch - 1) * p.block_table_stride + ((p.page_block_size & (p.page_block_size - 1)) == 0
                                        ? (p.seqlen_kv + p.page_block_size - 1) >> __builtin_ctz(p.page_block_size)
                                        : (p.seqlen_kv + p.page_block_size - 1) / p.page_block_size);
  const int table_ints = all_ints <= AE_WHOLE_TABLE ? (int)all_ints : AE_WHOLE_TABLE + 1;
  int table_all[AE_WHOLE_TABLE / 64];
  bool whole_table = false;
  int per_split = p.kv_per_split, n_mine = 0, len_b = 0;
  if (by_length) {
    if ((int)u >= p.tail_slots) return;                        // grid padding
    int len = lane < p.batch ? p.seqlens_k[lane] : 0;
    // a small block table is requested whole, together with the lengths (what an entry left unset is read, but never followed);
    // of a larger one the split's part, once it is known which that is: another trip to memory
    whole_table = table_ints <= AE_WHOLE_TABLE;
    if (whole_table && requests) {
#pragma unroll
      for (int i = 0; i < AE_WHOLE_TABLE / 64; i++)
        if (i * 64 + lane < table_ints) table_all[i] = p.block_table[i * 64 + lane];
    }
    len = len < p.seqlen_kv ? len : p.seqlen_kv;
    len = len > 0 ? len : 0;
    const ae_paged_splits s = ae_split_by_length(p, lane, (len + AE_BN - 1) / AE_BN);
    b = __builtin_popcountll(__builtin_amdgcn_ballot_w64(s.upto <= (int)u));     // entries in front of the unit's
    b = b < p.batch ? b : p.batch;
    if (b >= p.batch) return;                                  // (fewer splits than units)
    n_mine = __builtin_amdgcn_readlane(s.mine, b);
    split = (int)u - (__builtin_amdgcn_readlane(s.upto, b) - n_mine);
    per_split = s.tiles * AE_BN;
    len_b = __builtin_amdgcn_readlane(len, b);
    // (for the merge kernel: behind the row scales)
    if (split == 0 && ht == 0 && tid == 0)
      ((int*)(p.partial_rs + (int64_t)AE_N_ROWSCALES * p.batch * p.heads_q * n_split))[b] = n_mine;
  } else
#else
  const int per_split = p.kv_per_split;
#endif
  if (__builtin_expect(p.units_reciprocal != 0, 1)) {
    b = (int)(((uint64_t)u * (uint32_t)p.units_reciprocal) >> 32);
    split = (int)u - b * units;
  } else {
    b = ae_divide((int)u, units, split);
  }
#endif
  if (b >= p.batch * p.heads_kv || split >= n_split) return;  // grid padding (whole workgroup exits)
  if (AE_NSPLIT > 1 && !AE_PAGED && n_split < 2) return;      // (a launch for the build that writes out)
  if (__builtin_expect(p.heads_kv != 1, 0)) {
    hk = b % p.heads_kv;
    b /= p.heads_kv;
  }

  // (wave-uniform values are pinned to scalar registers: a copy in a vector register that gets spilled is
  // reloaded with a scratch load, which the tile loads' vmcnt bookkeeping would have to wait for)
  const int kv_begin = __builtin_amdgcn_readfirstlane(split * per_split);
#if AE_PAGED
  const ae_elem* k1 = (const ae_elem*)p.k + (int64_t)hk * p.k_stride_h;
  const ae_elem* k2 = (const ae_elem*)p.k2 + (int64_t)hk * p.k2_stride_h;
  const int32_t* pages = p.block_table + (int64_t)b * p.block_table_stride;
  const int page_size = p.page_block_size;
  int rq_slot0, top_slot;          // table slots of the split's first token and of the last one that it could hold
  {
    const int limit = by_length ? len_b : p.seqlen_kv;
    int top = kv_begin + per_split;
    top = (top < limit ? top : limit) - 1;
    top = top > 0 ? top : 0;
    if (__builtin_expect((page_size & (page_size - 1)) != 0, 0)) {
      rq_slot0 = kv_begin / page_size;
      top_slot = top / page_size;
    } else {
      rq_slot0 = kv_begin >> __builtin_ctz(page_size);
      top_slot = top >> __builtin_ctz(page_size);
    }
  }
  // The entry's length and the split's first 64 table entries are requested together (one after the other they held the
  // first tile back by another trip to memory).  So the entries are those that the split COULD hold: inside the table's
  // row; what an entry shorter than that left unset is read, but never followed.
  int seqlen_b = by_length ? len_b : p.seqlens_k[b];
  int table0 = 0;
  if (requests && !whole_table && rq_slot0 + lane <= top_slot) table0 = pages[rq_slot0 + lane];
#else
  const ae_elem* k1 = (const ae_elem*)p.k + (int64_t)b * p.k_stride_b + (int64_t)hk * p.k_stride_h;
  const ae_elem* k2 = (const ae_elem*)p.k2 + (int64_t)b * p.k2_stride_b + (int64_t)hk * p.k2_stride_h;
  const int seqlen_b = p.seqlen_kv;
#endif

#if AE_PAGED
  asm volatile("" ::: "memory");   // (both requests stay in front of the first wait and of the exits below)
#endif

  // ============================== tile requests =========================================================
  // Direct HBM -> LDS tile load, by the four value waves or by waves of their own: wave w fills AE_LOADS consecutive 1 KiB blocks of
  // the tile, starting at block min(w*AE_LOADS, AE_BLOCKS-AE_LOADS) (the last wave overlaps its neighbour, so
  // every wave issues the same number of loads); LDS chunk c' of row r receives global chunk c' ^ f(r).
  // Which row and chunk a lane fetches never changes: its byte offset inside a tile is computed once (one
  // register per load) and added per tile to the tile's wave-uniform address in the latent or in the rope
  // tensor.  The loads of a wave go out as bursts, each behind a single write of M0 (see
  // ae_load_lds16_burst; the offsets carry the compensation for its immediate offsets).  Rows past the
  // end re-read the last row.  Tiles past the end are not requested, so the waits for a tile ask whether a newer one
  // is on its way (a split of four tiles asked for nine when every trip requested one, and waited for them at its end).
  const int loader = AE_LOADER_WAVES ? wave - 4 : wave < 4 ? wave - 2 : wave - 4;
  const int blk0 = loader * AE_LOADS < AE_BLOCKS - AE_LOADS ? loader * AE_LOADS : AE_BLOCKS - AE_LOADS;
  // (the row and chunk of load i are carried along, and their row's offset with them: a division and a multiplication
  // per load were a third of the instructions in front of the first request)
  const int stride1 = (int)p.k_stride_s * 2, stride2 = (int)p.k2_stride_s * 2;   // bytes per kv row
#if AE_PAGED
  unsigned ld_uoff[AE_LOADS];
#else
  const char* ld_ptr[AE_LOADS];
  unsigned ld_adv[AE_LOADS];
#endif
  auto set_up_requests = [&]() AE_LAMBDA {
    int ld_row = (blk0 * 64 + lane) / AE_CPR, ld_cp = (blk0 * 64 + lane) % AE_CPR;
#if AE_PAGED
    // Paged cache: the latent and the rope part are column ranges of ONE cache tensor (equal strides, the rope
    // columns rope_delta bytes behind the latent ones: checked by ae_mla_decode_fwd), so every load of a tile is
    // (the tile's wave-uniform address) + (an offset of the lane that never changes): scalar base + 32-bit offset
    // loads, no address arithmetic per tile at all.  Bases are passed 4 KiB low and the offsets 4 KiB high, so
    // that the offsets, which carry the compensation for the immediate offsets, stay >= 0.
    const int rope_off = (int)((const char*)k2 - (const char*)k1) - AE_CPR1 * 16;
    int ld_roff = ld_row * stride1 + 4096;
#else
    // Dense cache: the requests go tile by tile, so a lane keeps the source address of each of its loads for the
    // NEXT tile to request and adds the tile pitch after every request - two instructions per load and tile.
    // (Two waves share a SIMD here: address arithmetic of ~140 instructions per tile and wave, as a base + offset
    // form needs, made these waves, not the matrix pipe, set the pace of the whole workgroup.)
    const char* const ld_base1 = (const char*)k1 + (uint64_t)((unsigned)kv_begin * (uint64_t)(unsigned)stride1);
    const char* const ld_base2 = (const char*)k2 + (uint64_t)((unsigned)kv_begin * (uint64_t)(unsigned)stride2);
    int ld_roff1 = ld_row * stride1, ld_roff2 = ld_row * stride2 - AE_CPR1 * 16;
#endif
#pragma unroll
    for (int i = 0; i < AE_LOADS; i++) {
      const int c = ld_cp ^ AE_SWZ(ld_row);
      const bool rope = c >= AE_CPR1;
      // immediate offset of load i inside its burst
      const int burst = i < AE_LB(1) ? 0 : i < AE_LB(2) ? 1 : 2;
      const int imm = (i - AE_LB(burst) - (AE_LB(burst + 1) - AE_LB(burst)) / 2) * 1024;
#if AE_PAGED
      ld_uoff[i] = (unsigned)(c * 16 + ld_roff + (rope ? rope_off : 0) - imm);
#else
      ld_ptr[i] = (rope ? ld_base2 : ld_base1) + (int64_t)(c * 16 + (rope ? ld_roff2 : ld_roff1) - imm);
      ld_adv[i] = AE_BN * (unsigned)(rope ? stride2 : stride1);
#endif
      ld_cp += 64 % AE_CPR;
      const bool wrap = ld_cp >= AE_CPR;
      const int rows = 64 / AE_CPR + (wrap ? 1 : 0);
      ld_cp -= wrap ? AE_CPR : 0;
      ld_row += rows;
#if AE_PAGED
      ld_roff += 64 / AE_CPR * stride1 + (wrap ? stride1 : 0);
#else
      ld_roff1 += 64 / AE_CPR * stride1 + (wrap ? stride1 : 0);
      ld_roff2 += 64 / AE_CPR * stride2 + (wrap ? stride2 : 0);
#endif
    }
  };
#if AE_PAGED
  if (requests) {
    set_up_requests();                       // while the entry's length and the table are on their way
#pragma unroll
    for (int i = 0; i < AE_LOADS; i++) asm volatile("" : "+v"(ld_uoff[i]));
  }
  seqlen_b = seqlen_b < p.seqlen_kv ? seqlen_b : p.seqlen_kv;
  seqlen_b = __builtin_amdgcn_readfirstlane(seqlen_b > 0 ? seqlen_b : 0);
#endif

  int kv_end_ = kv_begin + per_split;
  kv_end_ = kv_end_ < seqlen_b ? kv_end_ : seqlen_b;
  const int kv_end = __builtin_amdgcn_readfirstlane(kv_end_);
  const int n_tiles = __builtin_amdgcn_readfirstlane(kv_end > kv_begin ? (kv_end - kv_begin + AE_BN - 1) / AE_BN : 0);
#if AE_PAGED
  // a split beyond this entry's length: nothing to read (its table entries may be unset) and nothing to write,
  // the merge passes it over; split 0 of an entry of length 0 writes that entry's "no keys" result
  if (n_tiles == 0) {
    if (split == 0) ae_mla_write_no_keys(p, b, hk, ht, group, tid);
    return;
  }
#endif
  // who writes `out`: this workgroup (a launch without splits; a paged entry whose keys all lie in split 0), or the
  // merge kernel from the splits' partial results
#if AE_NSPLIT == 1
  constexpr bool direct = true;
#elif AE_PAGED
  const bool direct = seqlen_b <= per_split;           // (one split with keys at most)
#else
  constexpr bool direct = false;
#endif
  if (!AE_LOADER_WAVES && !score_wave && (wave == 4 || wave == 5)) return;      // placeholders: they only steer the value waves onto SIMD 2, 3

#if AE_HPW != 64
  if (score_wave) {
    // ======================= score wave: 16 heads, 16 of the tile's 32 keys ==============================
    const int half = wave & 1;                 // which keys; waves 4, 5: the second 16 heads
    const int l16 = lane & 15;
    const int g = lane >> 4;
    const int hl = (wave >> 2) * 16 + l16;     // head in the workgroup
    const int head_in_group = ht * AE_HEADS_PER_WG + hl;
    const int hq = hk * group + (head_in_group < group ? head_in_group : 0);
    // Q^T fragments: B operand (n = head = lane%16, k = d = 32*ks + 8*(lane/16) + j)
    const ae_elem* q1 = (const ae_elem*)p.q + (int64_t)b * p.q_stride_b + (int64_t)hq * p.q_stride_h;
    const ae_elem* q2 = (const ae_elem*)p.q2 + (int64_t)b * p.q2_stride_b + (int64_t)hq * p.q2_stride_h;
    ae_elem8 qf[AE_NKS];
#pragma unroll
    for (int ks = 0; ks < AE_D1 / 32; ks++) qf[ks] = *(const ae_elem8*)(q1 + ks * 32 + g * 8);
#pragma unroll
    for (int ks = 0; ks < AE_D2 / 32; ks++) qf[AE_D1 / 32 + ks] = *(const ae_elem8*)(q2 + ks * 32 + g * 8);

    ae_rowstate st;
    ae_rowstate_init(st);
    float m2 = st.AE_SM_M * AE_LOG2E;   // running reference, log2 units: the same in both halves' waves
    float r_run = half == 0 && g == 0 ? st.AE_SM_R : 0.f;      // this lane's part of the row sum
    __builtin_amdgcn_s_waitcnt(AE_VMCNT(0));   // Q has landed
    __syncthreads();                           // tile 0 has landed

    // K fragment of k-step ks: row 16*half + lane%16, global chunk 4*ks + lane/16 (swizzled in its three low bits)
    const int k_row = half * 16 + l16;
    int k_base[2];
#pragma unroll
    for (int i = 0; i < 2; i++) k_base[i] = k_row * AE_KSTR + (((4 * i + g) ^ AE_SWZ(k_row)) << 4);
    // A trip multiplies tile n by Q^T, with the softmax of tile n - 1 between those MFMAs, and leaves the row maxima of
    // tile n for the other half's wave.  A lane's scores: head lane%16, keys 16*half + 4*(lane/16) + e.
    float xs[4], mx;
    ae_lds_f32* const mine = xmax + half * AE_HPW + hl;
    const ae_lds_f32* const other = xmax + (1 - half) * AE_HPW + hl;
    float mn, osc, rs;
    bool need;
    // the softmax of tile tp in pieces, piece f issued behind the MFMA of k-step f
    auto soft_slot = [&](int f, int tp, float mo) AE_LAMBDA {
      if (f == 4) {
        mx = __builtin_fmaxf(mx, mo) * (AE_SM_SCALE * AE_LOG2E);   // the scale is positive
        need = (mx - m2) > AE_TAU2;
        mn = need ? mx : m2;
        osc = need ? ae_exp2(m2 - mn) : 1.0f;
        m2 = mn;
        rs = 0.f;
      } else if (f >= 5 && f < 9) {
        xs[f - 5] = ae_exp2(__builtin_fmaf(xs[f - 5], AE_SM_SCALE * AE_LOG2E, -mn));
        rs += xs[f - 5];
      } else if (f == 9) {
        // P^T [head][slot]: a value wave's lane takes slots 8*(lane/16) .. +7, the keys 4*(lane/16) .. +3 of both halves
        ae_elem4 w;
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = (ae_elem)xs[i];
        *(__attribute__((address_space(3))) ae_elem4*)(pbuf + (tp & 1) * AE_P_BYTES + hl * AE_PSTR + 16 * g + 8 * half) = w;
      } else if (f == 10) {
        r_run = r_run * osc + rs;
        ae_lds_byte* xb = xbuf + (tp & 1) * AE_X_BYTES;
        if (half == 0) {
          if (g == 0) ((ae_lds_f32*)xb)[hl] = osc;
          const bool any = __builtin_amdgcn_ballot_w64(need) != 0;
          if (lane == 0) ((ae_lds_i32*)(xb + AE_HEADS_PER_WG * 4))[wave >> 2] = any ? 1 : 0;
        }
      }
    };
    static_assert(AE_NKS >= 11, "the softmax of a tile is spread over 11 k-steps");
    auto score_trip = [&](int tn, auto with_soft) AE_LAMBDA {
      constexpr bool SOFT = decltype(with_soft)::value;
      int ka[2];
#pragma unroll
      for (int i = 0; i < 2; i++) ka[i] = k_base[i] + (tn % AE_NSTAGE) * AE_STAGE_BYTES;
      auto read_kfrag = [&](int ks) AE_LAMBDA -> ae_elem8 {
        return *(const __attribute__((address_space(3))) ae_elem8*)(lds + ka[ks & 1] + (ks >> 1) * 128);
      };
      float mo = 0.f;
      if (SOFT) mo = other[((tn - 1) & 1) * (AE_XMAX_BYTES / 4)];
      ae_elem8 ring[AE_RING];
#pragma unroll
      for (int f = 0; f < AE_AHEAD; f++) ring[f] = read_kfrag(f);
      ae_f32x4 sacc[2];
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int r = 0; r < 4; r++) sacc[c][r] = 0.f;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = 0; f < AE_NKS; f++) {
        if (f + AE_AHEAD < AE_NKS) ring[(f + AE_AHEAD) % AE_RING] = read_kfrag(f + AE_AHEAD);
        sacc[f & 1] = ae_mfma16(ring[f % AE_RING], qf[f], sacc[f & 1]);
        if (SOFT) soft_slot(f, tn - 1, mo);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int r = 0; r < 4; r++) xs[r] = sacc[0][r] + sacc[1][r];
      if (__builtin_expect(kv_begin + tn * AE_BN + AE_BN > kv_end, 0)) {     // keys beyond the end of the range
        asm volatile("" ::: "memory");
        const int kvb = kv_begin + tn * AE_BN + 16 * half + 4 * g;
#pragma unroll
        for (int e = 0; e < 4; e++) xs[e] = kvb + e < kv_end ? xs[e] : AE_NEG_INF;
      }
      mx = ae_group_max(__builtin_fmaxf(__builtin_fmaxf(xs[0], xs[1]), __builtin_fmaxf(xs[2], xs[3])));
      if (g == 0) mine[(tn & 1) * (AE_XMAX_BYTES / 4)] = mx;
    };
    if (n_tiles > 0) score_trip(0, ae_const_bool<false>());
    __syncthreads();                             // end of trip 0: tile 1 has landed
    for (int tn = 1; tn < n_tiles; tn++) {
      score_trip(tn, ae_const_bool<true>());
      __syncthreads();                           // end of the trip: P of tile tn - 1 is handed over, tile tn + 1 has landed
    }
    if (n_tiles > 0) {                           // the last tile's softmax has no MFMAs to hide behind
      const float mo = other[((n_tiles - 1) & 1) * (AE_XMAX_BYTES / 4)];
#pragma unroll
      for (int f = 4; f < 11; f++) soft_slot(f, n_tiles - 1, mo);
      __syncthreads();
    }
    const float r_row = ae_group_sum(r_run);
    if (g == 0) {                                // final row state for the value waves
      fin[hl * AE_FIN + 1 + half] = r_row;
      if (half == 0) fin[hl * AE_FIN] = m2 * AE_LN2;
    }
    __syncthreads();
    return;
  }
#else
  if (score_wave) {
    // =============================== score wave: 32 heads ==============================================
    const int l32s = lane & 31;
    const int hfs = lane >> 5;
    const int head_in_group = ht * AE_HEADS_PER_WG + wave * 32 + l32s;
    const int hq = hk * group + (head_in_group < group ? head_in_group : 0);
    // Q^T fragments: B operand (n = head = lane%32, k = d = 16*ks + 8*(lane/32) + j)
    const ae_elem* q1 = (const ae_elem*)p.q + (int64_t)b * p.q_stride_b + (int64_t)hq * p.q_stride_h;
    const ae_elem* q2 = (const ae_elem*)p.q2 + (int64_t)b * p.q2_stride_b + (int64_t)hq * p.q2_stride_h;
    ae_elem8 qf[AE_NKS];
#pragma unroll
    for (int ks = 0; ks < AE_D1 / 16; ks++) qf[ks] = *(const ae_elem8*)(q1 + ks * 16 + hfs * 8);
#pragma unroll
    for (int ks = 0; ks < AE_D2 / 16; ks++) qf[AE_D1 / 16 + ks] = *(const ae_elem8*)(q2 + ks * 16 + hfs * 8);

    ae_rowstate st;
    ae_rowstate_init(st);
    float m2 = st.AE_SM_M * AE_LOG2E;   // running reference, log2 units
    float r_run = st.AE_SM_R;           // this lane's part of the row sum (a row lives in lanes l, l^32)

    // (the value waves request the tiles: this wave's registers are taken by Q^T)
    __builtin_amdgcn_s_waitcnt(AE_VMCNT(0));   // Q has landed
    __syncthreads();                           // tile 0 has landed

    // K fragment of k-step ks: row lane%32, global chunk 2*ks + lane/32.  The swizzle touches the three low
    // bits of the chunk number only, so a lane has four distinct offsets (ks % 4) and the rest is an immediate.
    int k_base[4];
#pragma unroll
    for (int i = 0; i < 4; i++) k_base[i] = l32s * AE_KSTR + (((2 * i + hfs) ^ AE_SWZ(l32s)) << 4);
    // A trip multiplies tile n by Q^T and, in the issue slots between those MFMAs, runs the softmax of tile
    // n - 1 (its raw scores wait in `xs`): the wave's matrix work and its softmax overlap instead of
    // following each other.  P of tile n - 1 is handed over by the barrier that ends trip n.
    ae_f32x16 xs;        // raw scores of the tile before the one being multiplied
#pragma unroll
    for (int r = 0; r < 16; r++) xs[r] = 0.f;
    // lane owns head lane%32 and kv rows 8*(e/4) + 4*(lane/32) + e%4 of a tile
    float mx, mn, osc, rs;
    bool need;
    ae_lds_byte* prow;
    ae_lds_byte* xb;
    // start of the softmax of tile tp: scores beyond the end of the range are taken out (ragged tail only)
    auto soft_begin = [&](int tp) AE_LAMBDA {
      // (xs holds raw scores: the scale is folded into the exponent; the softmax works on it in place)
      const bool tail = kv_begin + tp * AE_BN + AE_BN > kv_end;
      if (__builtin_expect(tail, 0)) {
        // the empty asm keeps this a branch: flattened into selects it costs 5 instructions per score
        // on every tile
        asm volatile("" ::: "memory");
        const int kvb = kv_begin + tp * AE_BN + 4 * hfs;
#pragma unroll
        for (int e = 0; e < 16; e++) xs[e] = (kvb + 8 * (e >> 2) + (e & 3) < kv_end) ? xs[e] : AE_NEG_INF;
      }
      mx = AE_NEG_INF;
      rs = 0.f;
      prow = pbuf + (tp & 1) * AE_P_BYTES + (wave * 32 + l32s) * AE_PSTR + (AE_VB == 32 ? 8 : 16) * hfs;
      xb = xbuf + (tp & 1) * AE_X_BYTES;
    };
    // the softmax of one tile in AE_NKS pieces, piece f issued behind the MFMA of k-step f
    auto soft_slot = [&](int f) AE_LAMBDA {
      if (f < 4) {
        mx = __builtin_fmaxf(__builtin_fmaxf(mx, xs[4 * f]), xs[4 * f + 1]);
        mx = __builtin_fmaxf(__builtin_fmaxf(mx, xs[4 * f + 2]), xs[4 * f + 3]);
      } else if (f == 4) {
        float hi;
        const float lo = ae_swap32_lo_hi(mx, hi);
        mx = __builtin_fmaxf(lo, hi) * (AE_SM_SCALE * AE_LOG2E);   // the scale is positive
      } else if (f == 5) {
        need = (mx - m2) > AE_TAU2;
        mn = need ? mx : m2;
        osc = need ? ae_exp2(m2 - mn) : 1.0f;
        m2 = mn;
      } else if (f < 22) {
        const int e = f - 6;
        xs[e] = ae_exp2(__builtin_fmaf(xs[e], AE_SM_SCALE * AE_LOG2E, -mn));
        rs += xs[e];
      } else if (f < 26) {
        const int rb = f - 22;
        ae_elem4 w;
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = (ae_elem)xs[4 * rb + i];
        // (P^T [head][key]; 16-wide blocks [head][slot]: a value wave's lane takes slots 8*g .. + 7, keys 4*g .. + 3 of either half)
        *(__attribute__((address_space(3))) ae_elem4*)(prow + (AE_VB == 32 ? 16 * rb : 32 * (rb & 1) + 8 * (rb >> 1))) = w;
      } else if (f == 26) {
        r_run = r_run * osc + rs;
        if (hfs == 0) ((ae_lds_f32*)xb)[wave * 32 + l32s] = osc;
        const bool any = __builtin_amdgcn_ballot_w64(need) != 0;
        if (lane == 0) ((ae_lds_i32*)(xb + AE_HEADS_PER_WG * 4))[wave] = any ? 1 : 0;
      }
    };
    static_assert(AE_NKS >= 27, "the softmax of a tile is spread over 27 k-steps");
    // S^T of tile tn into xs; with SOFT the softmax of tile tn - 1 rides along
    auto score_trip = [&](int tn, auto with_soft) AE_LAMBDA {
      constexpr bool SOFT = decltype(with_soft)::value;
      int ka[4];
#pragma unroll
      for (int i = 0; i < 4; i++) ka[i] = k_base[i] + (tn % AE_NSTAGE) * AE_STAGE_BYTES;
      // read AE_AHEAD fragments before the MFMA that uses them (the compiler on its own keeps one read
      // in flight, which leaves the LDS latency exposed)
      auto read_kfrag = [&](int ks) AE_LAMBDA -> ae_elem8 {
        return *(const __attribute__((address_space(3))) ae_elem8*)(lds + ka[ks & 3] + (ks >> 2) * 128);
      };
      ae_elem8 ring[AE_RING];
#pragma unroll
      for (int f = 0; f < AE_AHEAD; f++) ring[f] = read_kfrag(f);
      if (SOFT) soft_begin(tn - 1);
      // even / odd k-steps accumulate separately (two independent MFMA chains)
      ae_f32x16 sacc[2];
#pragma unroll
      for (int c = 0; c < 2; c++)
#pragma unroll
        for (int r = 0; r < 16; r++) sacc[c][r] = 0.f;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = 0; f < AE_NKS; f++) {
        if (f + AE_AHEAD < AE_NKS) ring[(f + AE_AHEAD) % AE_RING] = read_kfrag(f + AE_AHEAD);
        sacc[f & 1] = ae_mfma32(ring[f % AE_RING], qf[f], sacc[f & 1]);
        if (SOFT) soft_slot(f);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int r = 0; r < 16; r++) xs[r] = sacc[0][r] + sacc[1][r];
    };
    if (n_tiles > 0) score_trip(0, ae_const_bool<false>());
    __syncthreads();                             // end of trip 0: tile 1 has landed
    for (int tn = 1; tn < n_tiles; tn++) {
      score_trip(tn, ae_const_bool<true>());
      __syncthreads();                           // end of the trip: P of tile tn - 1 is handed over, tile tn + 1 has landed
    }
    if (n_tiles > 0) {                           // the last tile's softmax has no MFMAs to hide behind
      soft_begin(n_tiles - 1);
#pragma unroll
      for (int f = 0; f < 27; f++) soft_slot(f);
      __syncthreads();
    }
    // final row state for the value waves
    {
      float hi;
      const float lo = ae_swap32_lo_hi(r_run, hi);
      if (hfs == 0) {
        fin[(wave * 32 + l32s) * AE_FIN] = m2 * AE_LN2;
        fin[(wave * 32 + l32s) * AE_FIN + 1] = lo + hi;
      }
    }
    __syncthreads();
    return;
  }
#endif

#if AE_LOADER_WAVES
  if (requests) {
#endif
#if !AE_PAGED
  set_up_requests();
#else
  // Paged cache: page, and row inside it, of the tile the NEXT request reads (wave-uniform; requests go tile by
  // tile, so no division per tile).  The split's part of the block table is copied into LDS first and looked up
  // there: once the tile loads are in flight, a table entry read from memory comes back through the same counter
  // as they do (the compiler cannot use a scalar load behind the loads' asm statements), and waiting for it means
  // waiting for every tile requested so far - 0.190 against 0.170 ms for the dense cache at B128 H128 S4096,
  // 0.166 ms with the table in LDS.  Every value wave writes the same entries and reads them back itself (a wave's
  // LDS operations complete in order), so no barrier is needed.
  int rq_idx = 0;
#if AE_NSPLIT > 1
  if (whole_table) {
#pragma unroll
    for (int i = 0; i < AE_WHOLE_TABLE / 64; i++)
      if (i * 64 + lane < table_ints) ptab[i * 64 + lane] = table_all[i];
    // (the first page from the registers: what goes through LDS is there when the second is looked up)
    rq_idx = b * p.block_table_stride + rq_slot0;
    const int at = rq_idx >> 6;
    table0 = table_all[0];
#pragma unroll
    for (int i = 1; i < AE_WHOLE_TABLE / 64; i++) table0 = at == i ? table_all[i] : table0;
    table0 = __builtin_amdgcn_readlane(table0, rq_idx & 63);
  } else
#endif
  {
  if (rq_slot0 + lane <= top_slot) ptab[lane] = table0;
  for (int i = 64 + lane; i < AE_PTAB && rq_slot0 + i <= top_slot; i += 64) ptab[i] = pages[rq_slot0 + i];   // (<= AE_PTAB: checked by ae_mla_decode_fwd)
  }
  int rq_in_page = kv_begin - rq_slot0 * page_size;
  int rq_page = __builtin_amdgcn_readfirstlane(table0);
#endif
  // requests are made for t = 0, 1, 2, ... in this order
  auto load_tile = [&](int t_) AE_LAMBDA {
    const int t = __builtin_amdgcn_readfirstlane(t_);
    if (t >= n_tiles) return;                       // (wave-uniform)
    const int kv0 = kv_begin + t * AE_BN;
    ae_lds_byte* dst = lds + (t % AE_NSTAGE) * AE_STAGE_BYTES;
    const bool ragged = kv0 + AE_BN > seqlen_b;     // wave-uniform
#if AE_PAGED
    // the tile's page was looked up when the previous request went out (rq_*, below); kv0 < seqlen_b, so its
    // table entry is set, and an entry outside the cache is clamped
    int page = rq_page < 0 ? 0 : (rq_page < p.num_pages ? rq_page : p.num_pages - 1);
    page = __builtin_amdgcn_readfirstlane(page);
    const char* tile = (const char*)k1 + ((int64_t)page * p.k_stride_b + (int64_t)rq_in_page * p.k_stride_s) * 2 - 4096;
    unsigned o[AE_LOADS];
#pragma unroll
    for (int i = 0; i < AE_LOADS; i++) o[i] = ld_uoff[i];
    if (__builtin_expect(ragged, 0)) {                        // rows past the end re-read the last row
      int ln = lane;
      asm volatile("" : "+v"(ln)::"memory");                  // (keeps this ONE branch, out of the common path, rows and all)
#pragma unroll
      for (int i = 0; i < AE_LOADS; i++) {
        const int row = ((blk0 + i) * 64 + ln) / AE_CPR;
        int over = kv0 + row - (seqlen_b - 1);
        over = over > 0 ? over : 0;                           // <= row: the offset stays >= 0
        o[i] -= (unsigned)(over * stride1);
      }
    }
    auto burst = [&](auto which) AE_LAMBDA {
      constexpr int LO = AE_LB(which.value), N = AE_LB(which.value + 1) - LO;
      unsigned ob[8];
#pragma unroll
      for (int i = 0; i < 8; i++) ob[i] = o[LO + (i < N ? i : 0)];
      ae_load_lds16_burst_base<N>(tile, ob, dst + (blk0 + LO + N / 2) * 1024);
    };
#else
    const char* g[AE_LOADS];
#pragma unroll
    for (int i = 0; i < AE_LOADS; i++) g[i] = ld_ptr[i];
    if (__builtin_expect(ragged, 0)) {                        // rows past the end re-read the last row
      int ln = lane;
      asm volatile("" : "+v"(ln)::"memory");                  // (keeps this ONE branch, out of the common path, rows and all)
#pragma unroll
      for (int i = 0; i < AE_LOADS; i++) {
        const int row = ((blk0 + i) * 64 + ln) / AE_CPR, cp = ((blk0 + i) * 64 + ln) % AE_CPR;
        int over = kv0 + row - (seqlen_b - 1);
        over = over > 0 ? over : 0;
        g[i] -= over * ((cp ^ AE_SWZ(row)) >= AE_CPR1 ? stride2 : stride1);
      }
    }
    auto burst = [&](auto which) AE_LAMBDA {
      constexpr int LO = AE_LB(which.value), N = AE_LB(which.value + 1) - LO;
      const char* gb[8];
#pragma unroll
      for (int i = 0; i < 8; i++) gb[i] = g[LO + (i < N ? i : 0)];
      ae_load_lds16_burst<N>((const void* const*)gb, dst + (blk0 + LO + N / 2) * 1024);
    };
#endif
    burst(ae_const_int<0>());
    burst(ae_const_int<1>());
    if constexpr (AE_BURSTS == 3) burst(ae_const_int<2>());
#if !AE_PAGED
#pragma unroll
    for (int i = 0; i < AE_LOADS; i++) ld_ptr[i] += ld_adv[i];
#else
    rq_in_page += AE_BN;                                      // where the next request reads: an LDS lookup per new
    if (rq_in_page >= page_size) {                            // page, a whole trip before its result is used
      rq_in_page = 0;
      rq_idx++;
      if (t + 1 < n_tiles) rq_page = ptab[rq_idx];
    }
#endif
  };
  // end of trip n, in which the score waves multiplied tile n and the value waves read tile n - 1: tile n + 1 has landed when
  // only the newest request (tile n + 2) is outstanding; after the barrier everyone is done with tile n - 1, whose stage
  // takes the next request
  auto end_trip = [&](int n) AE_LAMBDA {
    if (n + 2 < n_tiles) __builtin_amdgcn_s_waitcnt(AE_VMCNT_LGKM0(AE_LOADS));   // ... and this trip's LDS reads have returned
    else __builtin_amdgcn_s_waitcnt(AE_VMCNT_LGKM0(0));     // (the last tile has been requested: nothing is newer)
    __syncthreads();
    load_tile(n + 3);
  };

  __builtin_amdgcn_s_waitcnt(AE_VMCNT(0));
#pragma unroll
  for (int t = 0; t < 3; t++) load_tile(t);
  if (n_tiles >= 3) __builtin_amdgcn_s_waitcnt(AE_VMCNT(2 * AE_LOADS));
  else if (n_tiles == 2) __builtin_amdgcn_s_waitcnt(AE_VMCNT(AE_LOADS));
  else __builtin_amdgcn_s_waitcnt(AE_VMCNT(0));
#if AE_LOADER_WAVES
    __syncthreads();
    for (int n = 0; n <= n_tiles + 1; n++) end_trip(n);      // (the barriers of the value waves' trips)
    return;
  }
  auto end_trip = [&](int) AE_LAMBDA {
    __builtin_amdgcn_s_waitcnt(AE_VMCNT_LGKM0(63));            // (the trip's LDS reads have returned)
    __syncthreads();
  };
#endif

  // ============================== value wave: AE_DVW value columns, AE_HPW heads =======================
#if AE_VB == 32
  const int lhd = lane & 31;       // the lane's head in a block of heads
  const int hf = lane >> 5;        // ... and which part of the block's rows
#else
  const int lhd = lane & 15;
  const int hf = lane >> 4;
#endif
  const int dvw = wave < 4 ? wave - 2 : wave - 4;   // waves 2, 3, 6, 7
#if AE_VB == 32
  typedef ae_f32x16 ae_acc;
#else
  typedef ae_f32x4 ae_acc;
#endif
  constexpr int NR = sizeof(ae_acc) / 4;
  ae_acc oacc[AE_NHB][AE_NDB];     // [head block][dv block]: O^T
#pragma unroll
  for (int hb = 0; hb < AE_NHB; hb++)
#pragma unroll
    for (int db = 0; db < AE_NDB; db++)
#pragma unroll
      for (int r = 0; r < NR; r++) oacc[hb][db][r] = 0.f;
  __syncthreads();
#if AE_CLOCK_STAMPS
  const unsigned long long ae_w1 = __builtin_amdgcn_s_memrealtime();     // tile 0 (and Q) have landed
#endif

#if AE_VB == 32
  // V^T fragment (k-step kk, dv block db): A[m = dv][k = kv]: lane i of a 16-lane group supplies the
  // address of row 16*kk + 8*hf + i/4 (+4 for slots 4..7), 8 bytes at value column
  // 32*db + 16*((lane%32)/16) + 4*(i%4), and receives column i of those four rows.  The swizzle of a
  // row's chunks touches the three low bits of the chunk number only, so a lane has four distinct
  // offsets (parity of db, first / second group of four rows) and everything else is an immediate.
  const int v_row = 8 * hf + ((lane & 15) >> 2);
  const int v_c0 = 2 * (lhd >> 4) + ((lane & 3) >> 1);
  const int v_half = (lane & 1) * 8;
  int v_base[2][2];     // [db & 1][row group]
#pragma unroll
  for (int par = 0; par < 2; par++)
#pragma unroll
    for (int rg = 0; rg < 2; rg++) {
      const int r = v_row + 4 * rg;
      v_base[par][rg] = r * AE_KSTR + ((((4 * par + v_c0) ^ AE_SWZ(r)) + 4 * AE_NDB * dvw) << 4) + v_half;
    }
  auto read_vfrag = [&](const int (&va)[2][2], int kk, int db) AE_LAMBDA -> ae_elem8 {
    const int imm = 16 * kk * AE_KSTR + (db >> 1) * 128;
    ae_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) ae_s16x4*)(
        lds + va[db & 1][0] + imm));
    ae_s16x4 hi2 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) ae_s16x4*)(
        lds + va[db & 1][1] + imm));
    return __builtin_bit_cast(ae_elem8, __builtin_shufflevector(lo, hi2, 0, 1, 2, 3, 4, 5, 6, 7));
  };

#else
  // V^T fragment of dv block db (16 columns, all 32 keys): A[m = dv][k]: k = 8*(lane/16) + j is key 4*(lane/16) + j of the
  // tile's first half (j < 4) or second half (the order in which the score waves leave P): the 16 rows of one transposed
  // read then lie in 16 different places of the swizzle, where rows 0-3 and 8-11 would share theirs.
  const int v_row = 4 * hf + (lhd >> 2);
  int v_base[4];        // [db & 3]; rows 16 apart share a permutation
#pragma unroll
  for (int i = 0; i < 4; i++)
    v_base[i] = v_row * AE_KSTR + ((((2 * i + ((lane & 3) >> 1)) ^ AE_SWZ(v_row)) + (AE_DVW / 8) * dvw) << 4) + (lane & 1) * 8;
  auto read_vfrag = [&](const int (&va)[4], int, int db) AE_LAMBDA -> ae_elem8 {
    const int imm = (db >> 2) * 128;
    ae_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) ae_s16x4*)(
        lds + va[db & 3] + imm));
    ae_s16x4 hi2 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) ae_s16x4*)(
        lds + va[db & 3] + imm + 16 * AE_KSTR));
    return __builtin_bit_cast(ae_elem8, __builtin_shufflevector(lo, hi2, 0, 1, 2, 3, 4, 5, 6, 7));
  };
#endif

  // A trip of a value wave: O^T += V^T P^T for tile n - 2 with the V^T fragments it holds in registers (PV),
  // and the fragments of tile n - 1 read from LDS into those registers as they fall free (RD) - the read
  // has a whole trip to complete, and tile n - 1's stage can take the next request when the trip ends.
  constexpr int NKK = AE_VB == 32 ? 2 : 1;      // k-steps over the tile's keys
  ae_elem8 vreg[NKK * AE_NDB];     // fragment f = (k-step f / AE_NDB, dv block f % AE_NDB)
#pragma unroll
  for (int f = 0; f < NKK * AE_NDB; f++) vreg[f] = (ae_elem8){};
  auto value_trip = [&](int n, auto with_pv, auto with_rd) AE_LAMBDA {
    constexpr bool PV = decltype(with_pv)::value;
    constexpr bool RD = decltype(with_rd)::value;
    // the lane's four fragment offsets inside tile n - 1's stage
#if AE_VB == 32
    int va[2][2];
#pragma unroll
    for (int i = 0; i < 4; i++) va[i >> 1][i & 1] = v_base[i >> 1][i & 1] + ((n - 1) % AE_NSTAGE) * AE_STAGE_BYTES;
#else
    int va[4];
#pragma unroll
    for (int i = 0; i < 4; i++) va[i] = v_base[i] + ((n - 1) % AE_NSTAGE) * AE_STAGE_BYTES;
#endif
    ae_elem8 pf[AE_NHB][NKK];
    if (PV) {
      const int t = n - 2;
      const ae_lds_byte* pb = pbuf + (t & 1) * AE_P_BYTES;
      const ae_lds_byte* xb = xbuf + (t & 1) * AE_X_BYTES;
      // rescale O for the heads whose reference moved (rare once the maxima have settled)
      const ae_lds_i32* flags = (const ae_lds_i32*)(xb + AE_HEADS_PER_WG * 4);
      if (__builtin_amdgcn_readfirstlane(flags[0] | flags[AE_NSB - 1]) != 0) {
#pragma unroll
        for (int hb = 0; hb < AE_NHB; hb++) {
          const float osc = ((const ae_lds_f32*)xb)[hb * AE_VB + lhd];
#pragma unroll
          for (int db = 0; db < AE_NDB; db++)
#pragma unroll
            for (int r = 0; r < NR; r++) oacc[hb][db][r] *= osc;
        }
      }
      // P^T fragments: B[k = kv = 16*kk + 8*hf + j][n = head = 32*hb + lhd] (16 heads a block: all 32 kv, k = 8*hf + j)
#pragma unroll
      for (int hb = 0; hb < AE_NHB; hb++)
#pragma unroll
        for (int kk = 0; kk < NKK; kk++)
          pf[hb][kk] = *(const __attribute__((address_space(3))) ae_elem8*)(
              pb + (hb * AE_VB + lhd) * AE_PSTR + 32 * kk + 16 * hf);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int f = 0; f < NKK * AE_NDB; f++) {
      if (PV) {
#pragma unroll
        for (int hb = 0; hb < AE_NHB; hb++)
#if AE_VB == 32
          oacc[hb][f % AE_NDB] = ae_mfma32(vreg[f], pf[hb][f / AE_NDB], oacc[hb][f % AE_NDB]);
#else
          oacc[hb][f] = ae_mfma16(vreg[f], pf[hb][0], oacc[hb][f]);
#endif
      }
      if (RD) vreg[f] = read_vfrag(va, f / AE_NDB, f % AE_NDB);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  end_trip(0);                                                     // trip 0: the score waves multiply tile 0
  value_trip(1, ae_const_bool<false>(), ae_const_bool<true>());    // trip 1: fragments of tile 0
  end_trip(1);
  for (int n = 2; n <= n_tiles; n++) {
    value_trip(n, ae_const_bool<true>(), ae_const_bool<true>());
    end_trip(n);
  }
  if (n_tiles > 0) {                                               // trip n_tiles + 1: the last tile's product
    value_trip(n_tiles + 1, ae_const_bool<true>(), ae_const_bool<false>());
    end_trip(n_tiles + 1);
  }
  __builtin_amdgcn_s_waitcnt(AE_VMCNT(0));   // (the last barrier also made the final (m, r) of every head visible)
#if AE_CLOCK_STAMPS
  const unsigned long long ae_w2 = __builtin_amdgcn_s_memrealtime();     // the last trip is done
#endif

  // (... of every value wave: the score waves have left, and the tile stages take the results)
  __syncthreads();
  ae_lds_byte* obuf = lds + dvw * (AE_HEADS_PER_WG * AE_DVW * 4);
  const int heads_left = group - ht * AE_HEADS_PER_WG;          // heads of the tile that exist
  const int heads_here = heads_left < AE_HEADS_PER_WG ? heads_left : AE_HEADS_PER_WG;
  // ---- per-split epilogue: lane owns head 32*hb + lhd, value columns AE_DVW*dvw + 32*db + 8*(r/4) + 4*hf + r%4
  //      (16 heads a block: head 16*hb + lhd, columns AE_DVW*dvw + 16*db + 4*hf + r)
#pragma unroll
  for (int hb = 0; hb < AE_NHB; hb++) {
    if (hb * AE_VB >= heads_here) break;                        // (wave uniform)
    const int hl = hb * AE_VB + lhd;
    const int head_in_group = ht * AE_HEADS_PER_WG + hl;
    const bool head_ok = head_in_group < group;
    const int hq = hk * group + (head_ok ? head_in_group : 0);
    ae_ctx ctx;
    ctx.b = b;
    ctx.h = hq;
    ctx.q_idx = 0;
    ctx.kv_base = 0;
    ae_custom cust;
    ae_load_custom(cust, p, ctx);
    ae_rowstate st;
    ae_rowstate_init(st);
    float o[AE_NO];
#pragma unroll
    for (int db = 0; db < AE_NDB; db++)
#pragma unroll
      for (int r = 0; r < NR; r++) o[db * NR + r] = oacc[hb][db][r];
    float frs[AE_N_ROWSCALES > 0 ? AE_N_ROWSCALES : 1];
    frs[0] = 0.f;
    if (n_tiles > 0) {
      st.AE_SM_M = fin[hl * AE_FIN];
      st.AE_SM_R = fin[hl * AE_FIN + 1];
      if (AE_FIN == 3) st.AE_SM_R += fin[hl * AE_FIN + 2];
      ae_epilogue<AE_NO>(o, st, frs, ctx, cust);
    } else {
#pragma unroll
      for (int e = 0; e < AE_NO; e++) o[e] = 0.f;
#pragma unroll
      for (int i = 0; i < AE_N_ROWSCALES; i++) frs[i] = AE_NEG_INF;
    }
    // row scales: this lane's own head
    if (head_ok && hf == 0 && dvw == 0) {
      const int64_t row = ((int64_t)b * p.heads_q + hq) * n_split + split;
#pragma unroll
      for (int i = 0; i < AE_N_ROWSCALES; i++) {
        if (!direct) p.partial_rs[(int64_t)i * p.batch * p.heads_q * n_split + row] = frs[i];
        else if (p.rowscale_out[i]) p.rowscale_out[i][(int64_t)b * p.heads_q + hq] = frs[i];
      }
    }
    // O leaves through LDS, a head's AE_DVW columns as one contiguous piece (512 bytes fp32, 256 bytes in the output
    // type).  Stored straight from the accumulators it is 16 (8) bytes of each of 64 heads per instruction: lines that
    // are written in eight pieces, which the L2 has to put together (partial results of B4 H128, 8 MB: 2.8 us a
    // workgroup).  The partial results are stored past the cache (nontemporal, and read so by the merge kernel): their
    // lines are read once, on another XCD; left dirty they are written back between the two launches and again when the
    // next call's stores meet them.  B4 H128 Skv2048: call 24.7 -> 20.2 us.  16-byte chunks of a row are exchanged by the head number, so neither side meets a bank twice.
    // (piece e of a lane, four columns: fp32 chunk at4, in the output type half at4 % 2 of chunk at4 / 2)
#pragma unroll
    for (int e = 0; e < AE_NO / 4; e++) {
#if AE_VB == 32
      const int at4 = e * 2 + hf;                   // (dv block e / 4)
#else
      const int at4 = e * 4 + hf;
#endif
      if (direct) {
        ae_elem4 w;
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = (ae_elem)o[e * 4 + i];
        *(__attribute__((address_space(3))) ae_elem4*)(obuf + hl * (AE_DVW * 2) + (((at4 >> 1) ^ (hl & AE_OSW)) << 4) + (at4 & 1) * 8) = w;
      } else {
        const ae_f32x4 w = {o[e * 4 + 0], o[e * 4 + 1], o[e * 4 + 2], o[e * 4 + 3]};
        *(__attribute__((address_space(3))) ae_f32x4*)(obuf + hl * (AE_DVW * 4) + ((at4 ^ (hl & AE_OSW)) << 4)) = w;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (the wave's own region: its LDS writes have been made)
    // (the heads of a block leave while the next block's results are scaled and written)
    if (direct) {
      constexpr int CPH = AE_DVW / 8, N = AE_VB * CPH / 64;      // 16-byte chunks of a head's piece, instructions of the block
      ae_elem* ob = (ae_elem*)p.out + (int64_t)b * p.o_stride_b + (int64_t)(hk * group + ht * AE_HEADS_PER_WG) * p.o_stride_h + dvw * AE_DVW;
#pragma unroll 4
      for (int i = 0; i < N && i * 64 < (heads_here - hb * AE_VB) * CPH; i++) {
        const int hs = hb * AE_VB + (i * 64 + lane) / CPH, c = (i * 64 + lane) % CPH;
        const ae_elem8 w = *(const __attribute__((address_space(3))) ae_elem8*)(obuf + hs * (AE_DVW * 2) + ((c ^ (hs & AE_OSW)) << 4));
        if (hs < heads_here) *(ae_elem8*)(ob + (int64_t)hs * p.o_stride_h + c * 8) = w;
      }
    } else {
      constexpr int CPH = AE_DVW / 4, N = AE_VB * CPH / 64;
      float* ob = p.partial_o + (((int64_t)b * p.heads_q + hk * group + ht * AE_HEADS_PER_WG) * n_split + split) * AE_DV + dvw * AE_DVW;
#pragma unroll 8
      for (int i = 0; i < N && i * 64 < (heads_here - hb * AE_VB) * CPH; i++) {
        const int hs = hb * AE_VB + (i * 64 + lane) / CPH, c = (i * 64 + lane) % CPH;
        const ae_f32x4 w = *(const __attribute__((address_space(3))) ae_f32x4*)(obuf + hs * (AE_DVW * 4) + ((c ^ (hs & AE_OSW)) << 4));
        if (hs < heads_here) __builtin_nontemporal_store(w, (ae_f32x4*)(ob + (int64_t)hs * n_split * AE_DV + c * 4));
      }
    }
  }
#if AE_CLOCK_STAMPS
  __builtin_amdgcn_s_waitcnt(0);          // the stores have been acknowledged
  if (wave == 2) {
    const unsigned long long t1 = __builtin_amdgcn_s_memtime();
    const unsigned long long w1 = __builtin_amdgcn_s_memrealtime();
    if (lane == 0) {
      unsigned long long* st = (unsigned long long*)p.partial_o + 2 * (unsigned long long)blockIdx.x;
      st[0] = t1 - ae_t0;
      st[1] = w1 - ae_w0;
      unsigned long long* ph = (unsigned long long*)p.partial_o + 2 * (unsigned long long)gridDim.x +
                               4 * (unsigned long long)blockIdx.x;
      ph[0] = ae_w0;
      ph[1] = ae_w1;
      ph[2] = ae_w2;
      ph[3] = w1;
    }
  }
#endif
}

#ifdef AE_COMBINE_THREADS       // (a caller that wants both kernels in one module)
#include "ae_combine.h"
#endif
