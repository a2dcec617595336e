// Merge kernel of the split-KV launches (ae_decode.hip, ae_mla_decode.hip, ae_mla_decode_ws.hip, ae_prefill.hip).
//
// Needs AE_DV, AE_N_ROWSCALES, AE_COMBINE_THREADS, AE_NSPLIT (the most partial results of a row that the build merges),
// AE_SPLITS_PER_PARTIAL (splits of the launch that a partial result holds: the waves of a workgroup that merged theirs first,
// else 1) and the generated ae_combine().
//
// Built as a module of its own (ae_combine.hip): the split kernels take the number of splits from the launch and are built
// once; this one holds the weights of a row in registers and is built for 2, 4, 8 ... 64 partial results.  Places beyond the launch's count hold zero
// and weigh nothing, as the splits beyond a paged entry's length do.  (Built together for every count, a cache
// that grew from 256 to 8192 tokens met up to 37 builds of 0.8 s.)

#ifndef AE_COMBINE_H
#define AE_COMBINE_H

#ifndef AE_SPLITS_PER_PARTIAL
#define AE_SPLITS_PER_PARTIAL 1
#endif
#define AE_COMBINE_ROWS (AE_COMBINE_THREADS / (AE_DV / 4) > 0 ? AE_COMBINE_THREADS / (AE_DV / 4) : 1)
static_assert(AE_DV % 4 == 0, "four value columns a thread");

template <int N> struct ae_places { static constexpr int value = N; };

// Merge of the per-split partials: grid (ceil(Hq / AE_COMBINE_ROWS), B).  Bound by its chain of dependent memory
// trips (row scales, then partial results), not by bytes, so a thread owns four neighbouring value columns (16-byte
// loads, one pass over DV 512 with 128 threads where one column a thread took four) and a workgroup holds as many
// rows as its threads have room for (ae_tile_cfg.block_m of the combine configuration).
// out[b,0,h,:] = sum_k partial_o[b,h,k,:] * o_scale[k], o_scale = combine(final_rowscales[k])
// (attn_gqa_decode_tl.py:224-266; generic form core/template/tl_template/attn/attn_decode_tl.py:184-189).
extern "C" __global__ __launch_bounds__(AE_COMBINE_THREADS)
void ae_decode_combine_kernel(const ae_attn_params p) {
  constexpr int TPR = AE_DV / 4 < AE_COMBINE_THREADS ? AE_DV / 4 : AE_COMBINE_THREADS;      // threads per row
  const int h = AE_COMBINE_ROWS == 1 ? blockIdx.x : blockIdx.x * AE_COMBINE_ROWS + threadIdx.x / TPR;
  const int b = blockIdx.y;
  const int n_part = (unsigned)p.num_splits / AE_SPLITS_PER_PARTIAL;
  if (threadIdx.x >= AE_COMBINE_ROWS * TPR || h >= p.heads_q) return;
  // Paged cache (per-entry lengths): only the first ceil(length / kv_per_split) splits of an entry hold keys and
  // wrote partial results; an entry with at most one wrote `out` itself.
  int n_used = n_part;
  if (p.seqlens_k != nullptr) {
    if (p.tail_slots != 0) {           // (the split kernel has cut the entries, and says how often)
      n_used = ((const int*)(p.partial_rs + (int64_t)AE_N_ROWSCALES * p.batch * p.heads_q * n_part))[b];
    } else {
      int len = p.seqlens_k[b];
      len = len < p.seqlen_kv ? len : p.seqlen_kv;
      const int n = (int)((unsigned)((len > 0 ? len : 0) + p.kv_per_split - 1) / (unsigned)p.kv_per_split);
      n_used = n < n_part ? n : n_part;
    }
    if (n_used <= 1) return;
  }
  // The partial results are read 16 splits at a time, unconditionally, so that the loads of a group all go
  // out before the first one is waited for (one memory round trip per group instead of one per split: the
  // merge of 32 splits 18 -> 4 us).  The row scales are read the same way, in front of the first group, whose weights they
  // are: one trip to memory for both (B8 H128, paged, 16 splits: the call 22.2 -> 21.5 us).  Places without a result
  // have a row scale of -inf and lie behind the buffer's end, where a result reads as zero (not as another one once more: zero
  // times infinity is no number).  `places`: the number of results where it is one of those that the dispatch below knows, a
  // constant then and no place is empty (B36 H16, paged, 5 of 8 places: merge 3.36 us, 3.70 with comparisons); 0 for others.
  const int row_here = AE_COMBINE_ROWS == 1 ? 0 : threadIdx.x / TPR;
  const int rows_left = p.heads_q - blockIdx.x * AE_COMBINE_ROWS;
  const int64_t row0 = ((int64_t)b * p.heads_q + blockIdx.x * AE_COMBINE_ROWS) * n_part;       // the workgroup's rows are contiguous
  // (pinned to a scalar register: in a vector register every load would loop over the lanes' descriptors)
  const int row_bytes = __builtin_amdgcn_readfirstlane(AE_COMBINE_ROWS == 1 ? n_used * 4 : (rows_left < AE_COMBINE_ROWS ? rows_left : AE_COMBINE_ROWS) * n_part * 4);
  auto merge = [&](auto places) AE_LAMBDA {
    constexpr bool kFixed = decltype(places)::value > 0;
    constexpr int N = kFixed ? decltype(places)::value : AE_NSPLIT, G = N < 16 ? N : 16;
    // (the count is compared as a vector register, a copy for each use: 64 scalar conditions, or the results of as many
    // vector ones kept from one use to the next, do not fit the scalar registers)
    int n_row = n_used, n_load = n_used, n_weight = n_used, n_sum = n_used;
    if (!kFixed) asm volatile("" : "+v"(n_row), "+v"(n_load), "+v"(n_weight), "+v"(n_sum));
    int row_at = row_here * n_part * 4;
    asm volatile("" : "+v"(row_at));       // (one register, the places as offsets in the instructions)
    __amdgpu_buffer_rsrc_t part = __builtin_amdgcn_make_buffer_rsrc(p.partial_o + row0 * AE_DV, 0, row_bytes * AE_DV, 0x00020000);
    auto load_group = [&](ae_f32x4 (&val)[G], int k0, int dv) AE_LAMBDA {
#pragma unroll
      for (int i = 0; i < G; i++) {
        const int k = k0 + i;
        const bool there = kFixed ? k < N : AE_COMBINE_ROWS == 1 || k < n_load;
        // (read once: past the caches, see ae_mla_decode_ws.hip)
        constexpr int kNonTemporal = 2;
        val[i] = __builtin_bit_cast(ae_f32x4, __builtin_amdgcn_raw_buffer_load_b128(
            part, there ? row_at * AE_DV + dv * 4 + k * (AE_DV * 4) : -1, 0, kNonTemporal));
      }
    };
    const int dv0 = (threadIdx.x % TPR) * 4;
    float rs[AE_N_ROWSCALES > 0 ? AE_N_ROWSCALES : 1][N];
#pragma unroll
    for (int i = 0; i < AE_N_ROWSCALES; i++) {
      __amdgpu_buffer_rsrc_t scales = __builtin_amdgcn_make_buffer_rsrc(
          p.partial_rs + (int64_t)i * p.batch * p.heads_q * n_part + row0, 0, row_bytes, 0x00020000);
#pragma unroll
      for (int k = 0; k < N; k++)
        rs[i][k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(scales, row_at + (kFixed || k < n_row ? k : 0) * 4, 0, 0));
    }
    ae_f32x4 val[G];
    load_group(val, 0, dv0);
    __builtin_amdgcn_sched_barrier(0);             // (left alone the compiler moves the loads behind the weights)
    if (!kFixed) {
#pragma unroll
      for (int i = 0; i < AE_N_ROWSCALES; i++)
#pragma unroll
        for (int k = 0; k < N; k++) rs[i][k] = k < n_weight ? rs[i][k] : AE_NEG_INF;
    }
    float w[N];
    float merged[AE_N_ROWSCALES > 0 ? AE_N_ROWSCALES : 1];
    ae_combine(rs, w, merged);
    ae_elem* optr = (ae_elem*)p.out + (int64_t)b * p.o_stride_b + (int64_t)h * p.o_stride_h;
    for (int dv = dv0; dv < AE_DV; dv += TPR * 4) {
      if (dv != dv0) load_group(val, 0, dv);
      ae_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k0 = 0; k0 < N; k0 += G) {
        if (k0) load_group(val, k0, dv);
#pragma unroll
        for (int i = 0; i < G; i++) {
          const int k = k0 + i;
          const float wk = k < N && (kFixed || k < n_sum) ? w[k < N ? k : 0] : 0.f;
#pragma unroll
          for (int c = 0; c < 4; c++) acc[c] += val[i][c] * wk;
        }
      }
      ae_elem4 r;
#pragma unroll
      for (int c = 0; c < 4; c++) r[c] = (ae_elem)acc[c];
      *(ae_elem4*)(optr + dv) = r;
    }
    if (threadIdx.x % TPR == 0) {
      // One-token decode: row scales [B, Hq].  Split-KV prefill (p.seqlen_q > 1: its launch hands the (q position,
      // head) pairs over as p.heads_q = Sq * Hq "heads", h = s * Hq + head): row scales [B, Hq, Sq], the layout of
      // the unsplit kernels.
      int64_t at = (int64_t)b * p.heads_q + h;
      if (p.seqlen_q > 1) {
        const int hq = p.heads_q / p.seqlen_q;
        at = ((int64_t)b * hq + h % hq) * p.seqlen_q + h / hq;
      }
#pragma unroll
      for (int i = 0; i < AE_N_ROWSCALES; i++)
        if (p.rowscale_out[i]) p.rowscale_out[i][at] = merged[i];
    }
  };
  if (__builtin_expect(n_used == AE_NSPLIT, 1)) merge(ae_places<AE_NSPLIT>());
#if AE_NSPLIT % 4 == 0
  else if (n_used == AE_NSPLIT / 4 * 3) merge(ae_places<AE_NSPLIT / 4 * 3>());
#endif
#if AE_NSPLIT % 8 == 0
  else if (n_used == AE_NSPLIT / 8 * 5) merge(ae_places<AE_NSPLIT / 8 * 5>());
  else if (n_used == AE_NSPLIT / 8 * 7) merge(ae_places<AE_NSPLIT / 8 * 7>());
#endif
#if AE_NSPLIT == 8 || AE_NSPLIT == 16
  else if (n_used == AE_NSPLIT / 2) merge(ae_places<AE_NSPLIT / 2>());       // (paged entries have any count)
  else if (n_used == AE_NSPLIT / 8 * 3) merge(ae_places<AE_NSPLIT / 8 * 3>());
  else if (n_used == AE_NSPLIT / 4) merge(ae_places<AE_NSPLIT / 4>());
#endif
#if AE_NSPLIT == 16
  else if (n_used == 9) merge(ae_places<9>());
  else if (n_used == 11) merge(ae_places<11>());
  else if (n_used == 13) merge(ae_places<13>());
  else if (n_used == 15) merge(ae_places<15>());
#endif
  else merge(ae_places<0>());
}

#endif  // AE_COMBINE_H
