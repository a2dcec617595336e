// Merge of a split launch by the workgroup that finishes last (ae_prefill.hip; ae_decode.hip has its own).  Every workgroup stores its partial
// results with device scope (the merging one may sit on another XCD), waits for them, then counts itself in on a counter of
// its rows, behind the row scales in p.partial_rs; the last one sets the counter back to zero and merges.  Needs AE_DV,
// AE_N_ROWSCALES == 1 and the generated ae_combine().
//
// Bound by the counter's trip to memory and the read of all partial results by one workgroup; the merge launch that it replaces
// takes 3 us and the gap in front of it.  It is only worth it for a few rows, see PrefillOp._merges_in_last.  The results are held in
// registers, 32 loads of 16 bytes a thread at once: through LDS, in loops that are short enough not to wait for their
// own code, the same 70 calls were 6 % slower on average (B4 H8 Sq15 Skv532 D128: 9.4 us, 11.6 through LDS).  The count is a
// constant (a switch over 2 to 8): built for 4 or 8 places, some of them empty, it gave sums in another order of rounding and
// 0.95 of the time of two launches on average, this 0.94.

#ifndef AE_MERGE_LAST_H
#define AE_MERGE_LAST_H

constexpr int kAeDeviceScope = 16;     // the sc1 bit of a buffer instruction's cache policy

// After the workgroup's partial results have been stored: true in the one that came last of `n`.  `flag`: a word of LDS that
// nobody reads or writes any more.
AE_DEV bool ae_count_in(int* counter, int n, bool elected, __attribute__((address_space(3))) int* flag) {
  __builtin_amdgcn_s_waitcnt(0x0F70);          // vmcnt(0): the stores have been acknowledged
  __syncthreads();
  if (elected) {
    const int last = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
    // (nobody else touches the counter until the next launch)
    if (last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = last;
  }
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(*flag) != 0;
}

// Rows 0 .. n_rows - 1 of N partial results each, the first one of row r `r * row_step` behind `first` (in the buffers of
// results and of row scales), by NT threads (t: this one's number), AE_DV / 4 of them a row: write(r, column, four columns,
// merged row scale).  Bit for bit what ae_decode_combine_kernel gives, which knows these counts as constants too: the same sums in the
// same order, contracted alike.
template <int NT, int N, class Write>
AE_DEV void ae_merge_rows(const ae_attn_params& p, int64_t first, int row_step, int t, int n_rows, Write write) {
  constexpr int TPR = AE_DV / 4, RP = NT / TPR, G = 32 / N;      // threads a row, rows a pass, passes in flight
  static_assert(NT % TPR == 0 && AE_N_ROWSCALES == 1, "whole rows a pass, one row scale");
  const int n_buffer = (n_rows - 1) * row_step + N;
  __amdgpu_buffer_rsrc_t part = __builtin_amdgcn_make_buffer_rsrc(p.partial_o + first * AE_DV, 0, n_buffer * AE_DV * 4, 0x00020000);
  __amdgpu_buffer_rsrc_t scales = __builtin_amdgcn_make_buffer_rsrc(p.partial_rs + first, 0, n_buffer * 4, 0x00020000);
  const int col = t % TPR * 4;
  for (int r0 = 0; r0 < n_rows; r0 += RP * G) {
    float rs[G][1][N];
    ae_f32x4 val[G][N];
    // (rows that are not there are read behind the buffers' end, which takes no trip to memory)
#pragma unroll
    for (int g = 0; g < G; g++) {
      const int r = r0 + t / TPR + g * RP, at = r * row_step;
#pragma unroll
      for (int k = 0; k < N; k++) {
        rs[g][0][k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(scales, r < n_rows ? (at + k) * 4 : -1, 0, kAeDeviceScope));
        val[g][k] = __builtin_bit_cast(ae_f32x4, __builtin_amdgcn_raw_buffer_load_b128(
            part, r < n_rows ? ((at + k) * AE_DV + col) * 4 : -1, 0, kAeDeviceScope));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < G; g++) {
      const int r = r0 + t / TPR + g * RP;
      float w[N], merged[1];
      ae_combine(rs[g], w, merged);
      ae_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < N; k++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[c] += val[g][k][c] * w[k];
      if (r < n_rows) write(r, col, acc, merged[0]);
    }
  }
}

template <int NT, class Write>
AE_DEV void ae_merge_rows(const ae_attn_params& p, int64_t first, int row_step, int t, int n_rows, int n_used, Write write) {
  switch (n_used) {
    case 2: ae_merge_rows<NT, 2>(p, first, row_step, t, n_rows, write); break;
    case 3: ae_merge_rows<NT, 3>(p, first, row_step, t, n_rows, write); break;
    case 4: ae_merge_rows<NT, 4>(p, first, row_step, t, n_rows, write); break;
    case 5: ae_merge_rows<NT, 5>(p, first, row_step, t, n_rows, write); break;
    case 6: ae_merge_rows<NT, 6>(p, first, row_step, t, n_rows, write); break;
    case 7: ae_merge_rows<NT, 7>(p, first, row_step, t, n_rows, write); break;
    default: ae_merge_rows<NT, 8>(p, first, row_step, t, n_rows, write);
  }
}

#endif
