// Device-side helpers shared by the gfx950 attention kernel templates.
//
// Element types, MFMA wrappers, the register layouts of the 32x32x16 MFMA accumulator and
// the row reductions / transcendentals the generated functors call. The transcendental
// definitions follow the reference's code generator (core/codegen/tl_gen.py:89-117):
// exp(x) = exp2(x * log2 e), log(x) = log2(x) * ln 2, tanh via a fast approximation.
#ifndef AE_DEVICE_H
#define AE_DEVICE_H

// hipRTC predefines the HIP device environment; an offline hipcc build has to include it.
#ifndef __HIPCC_RTC__
#include <hip/hip_runtime.h>
#endif
#include "ae_hip.h"

#if AE_DTYPE_BF16
typedef __bf16 ae_elem;
#else
typedef _Float16 ae_elem;
#endif
typedef ae_elem ae_elem8 __attribute__((ext_vector_type(8)));
typedef ae_elem ae_elem4 __attribute__((ext_vector_type(4)));
typedef ae_elem ae_elem2 __attribute__((ext_vector_type(2)));
typedef float ae_f32x16 __attribute__((ext_vector_type(16)));
typedef float ae_f32x4 __attribute__((ext_vector_type(4)));
typedef short ae_s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int ae_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int ae_u32x2 __attribute__((ext_vector_type(2)));

#define AE_DEV __device__ inline __attribute__((always_inline))
// for the call operator of a lambda: a lambda that the inliner leaves as a function keeps the arrays it captures
// by reference in scratch memory (seen with the larger bf16 builds of the pipelined prefill kernel: 752 bytes of
// scratch per lane, 30 times the run time)
#define AE_LAMBDA __attribute__((always_inline))
#define AE_NEG_INF (-__builtin_inff())
#define AE_LOG2E 1.4426950408889634f
#define AE_LN2 0.6931471805599453f

// Quotient and remainder of wave-uniform numbers, a >= 0 and d > 0.  The compiler's division is a chain of some thirty
// dependent instructions, and which tile a workgroup has takes four of them in front of its first request: a shift where d
// is a power of two, else a reciprocal, whose quotient is off by at most one below 2^22 (three roundings, 2^-22 of it together).
AE_DEV int ae_divide_small(int a, int d, int& rem) {       // a below 2^31, a / d below 2^22
  int q = __builtin_amdgcn_readfirstlane((int)((float)a * __builtin_amdgcn_rcpf((float)d)));
  rem = a - q * d;
  if (rem < 0) q--, rem += d;
  if (rem >= d) q++, rem -= d;
  return q;
}
AE_DEV int ae_divide(int a, int d, int& rem) {
  int q;
  if ((d & (d - 1)) == 0) {
    q = a >> __builtin_ctz(d);
    rem = a & (d - 1);
  } else if (__builtin_expect(a < 1 << 22, 1)) {
    // (ae_divide_small, written out: with a call of it the compiler lays the latent decode out differently, B8 H128 of 2048 tokens,
    // paged, 18.55 -> 18.75 us)
    q = __builtin_amdgcn_readfirstlane((int)((float)a * __builtin_amdgcn_rcpf((float)d)));
    rem = a - q * d;
    if (rem < 0) q--, rem += d;
    if (rem >= d) q++, rem -= d;
  } else {
    q = a / d;
    rem = a - q * d;
  }
  return q;
}

// Which head and which tile a workgroup has.  Consecutive ids are dealt round-robin to the 8 XCDs, each with an L2 of 4 MB of
// its own, so the workgroups of id 8 * slot + xcd share one.
// ae_head_of_xcd: the (batch, query head) whose turn among the heads of its XCD is i; n_bh or more: none.  in_runs (launches whose
// query heads share kv heads): an XCD has neighbouring heads, so that K and V of fewer kv heads go through its L2; else turn i
// of the eight XCDs are eight neighbours, whose rows lie side by side in memory.  us, dealt singly -> in runs: causal bf16 B4 Hq64
// Hkv8 D128 S1000 104.3 -> 88.8, S2000 348 -> 291, fp16 S333 26.3 -> 22.9, B4 Hq32 Hkv8 S3000 D64 181.8 -> 172.5, B2 Hq32 Hkv8 S4096
// D128 275.5 -> 270.7, without a mask B1 Hq64 Hkv8 S700 25.0 -> 24.6, forward and backward of B8 Hq32 Hkv8 S1500 D64 451 -> 432.
// (Heads with K and V of their own in runs: 0.99 to 1.015.)
// With fewer than eight heads an XCD (AE_RUNS_FROM) the whole K and V fit every L2, and one head's lines asked for by all workgroups of
// an XCD are late: B1 Hq32 Hkv8 S333 with inputs in the caches 8.77 -> 8.95 (not in them 9.19 -> 8.97); B1 Hq64 Hkv8 S333 10.87 ->
// 10.71 (11.69 -> 11.25).
#define AE_RUNS_FROM 8
AE_DEV int ae_head_of_xcd(int i, int xcd, int n_bh, bool in_runs) {
  if (!in_runs) return i * 8 + xcd;
  const int lo = n_bh >> 3, more = n_bh & 7;
  return i < lo + (xcd < more ? 1 : 0) ? xcd * lo + (xcd < more ? xcd : more) + i : n_bh;
}
// ae_heavy_first: q tiles that differ in work, the tile with the most work first across the heads of the XCD (longest job first
// keeps the tail short).  Returns how many tiles of the head lie in front of it in that order; i: the head's turn.  in_eights: the
// first three quarters of the tiles go eight heads at a time - the tiles in flight are then of few heads, which keeps their K
// and V in the L2, and what is left for the end is short.  Pays where an XCD has more heads than that, each with K and V of its own, and
// more than two rounds of workgroups.  us, all heads -> eight at a time: causal 192 / 128 columns B1 H128 S2500 269 -> 265 (bf16), B2
// H128 S1400 208 -> 197 (fp16), B4 H128 S700 158 -> 133 (bf16); 128 columns, 128-row tiles, B8 H32 S875 87.5 -> 80.0, B4 H32 S2048 162.9 ->
// 159.8; 64 columns B8 H32 S1700 143 -> 135; 256-row tiles of the pipelined kernel, B4 H32 S4096 570 -> 557, S2500 249 -> 241.  Where
// there is less it costs: B1 H128 S400 (64 tiles an XCD) 19.7 -> 21.1, D64 B4 H32 S1200 (160) 39.6 -> 40.1.  Two or four heads at
// a time, or all tiles that way: up to 15 % worse at some lengths.  The launches of the backward: no difference beyond 1 %.
AE_DEV int ae_heavy_first(int slot, int n_bg, int n_t, bool in_eights, int& i) {
  if (in_eights) {
    const int n_long = n_t - n_t / 4;
    if (slot < n_long * n_bg) {
      int r;
      const int i0 = ae_divide_small(slot, 8 * n_long, r) * 8;
      int t = r >> 3;
      i = r & 7;
      if (n_bg - i0 < 8) t = ae_divide_small(r, n_bg - i0, i);
      i += i0;
      return t;
    }
  }
  return ae_divide(slot, n_bg, i);
}

// D[m][n] += sum_k A[m][k] B[k][n], 32x32 output, 16-deep. Lane l supplies A[l%32][8*(l/32)+j]
// and B[8*(l/32)+j][l%32], j=0..7, and owns D[8*(r/4) + 4*(l/32) + r%4][l%32], r=0..15.
AE_DEV ae_f32x16 ae_mfma32(ae_elem8 a, ae_elem8 b, ae_f32x16 c) {
#if AE_DTYPE_BF16
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
#else
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
#endif
}

// D[m][n], 16x16 output, 32-deep. Lane l supplies A[l%16][8*(l/16)+j], B[8*(l/16)+j][l%16]
// and owns D[4*(l/16) + r][l%16], r=0..3.
AE_DEV ae_f32x4 ae_mfma16(ae_elem8 a, ae_elem8 b, ae_f32x4 c) {
#if AE_DTYPE_BF16
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
#else
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
#endif
}

// ---- direct HBM -> LDS load --------------------------------------------------------------------
// 16 bytes per lane from `gptr` (any per-lane address) to LDS at lds_base + lane*16, lds_base wave
// uniform.  Issued as inline assembly rather than through __builtin_amdgcn_global_load_lds: when the
// compiler knows about a pending LDS-DMA write it makes every LDS read it cannot prove disjoint
// (all ds_read_tr*, which carry no precise memory operand) wait for vmcnt(0), i.e. for the tile that
// was just requested for LATER, which serialises the prefetch.  Callers order these loads against
// their consumers themselves: s_waitcnt vmcnt(..) followed by a workgroup barrier.
typedef __attribute__((address_space(3))) unsigned char ae_lds_u8;
AE_DEV void ae_load_lds16(const void* gptr, ae_lds_u8* lds_base) {
  const unsigned m0v = __builtin_amdgcn_readfirstlane((unsigned)(unsigned long)lds_base);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(gptr), "s"(m0v) : "memory");
}

// The 4-byte form: lane i's dword lands at lds_base + 4*i.
AE_DEV void ae_load_lds4(const void* gptr, ae_lds_u8* lds_base) {
  const unsigned m0v = __builtin_amdgcn_readfirstlane((unsigned)(unsigned long)lds_base);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(gptr), "s"(m0v) : "memory");
}

// N (1..8) such loads behind ONE write of M0.  Every write of M0 makes the wave wait for its LDS reads
// in flight, which costs a kernel that keeps its LDS pipe busy about 40 ns per load; a burst pays that
// once.  Load i lands at lds_mid + (i - N/2) KiB + lane*16.  The instruction's immediate offset moves
// the LDS address AND the global address, so the caller passes g[i] = source pointer - (i - N/2) KiB
// (the sum is what is dereferenced).  g must have 8 entries; those from N on are ignored.
template <int N>
AE_DEV void ae_load_lds16_burst(const void* const* g, ae_lds_u8* lds_mid) {
  static_assert(N >= 1 && N <= 8, "the 13-bit signed immediate offset reaches -4 KiB .. +3 KiB");
  const unsigned m0v = __builtin_amdgcn_readfirstlane((unsigned)(unsigned long)lds_mid);
  asm volatile(
      "s_mov_b32 m0, %8\n\ts_nop 0\n\t"
      "global_load_lds_dwordx4 %0, off offset:(0-%9/2)*1024\n\t"
      ".if %9 > 1\n\tglobal_load_lds_dwordx4 %1, off offset:(1-%9/2)*1024\n\t.endif\n\t"
      ".if %9 > 2\n\tglobal_load_lds_dwordx4 %2, off offset:(2-%9/2)*1024\n\t.endif\n\t"
      ".if %9 > 3\n\tglobal_load_lds_dwordx4 %3, off offset:(3-%9/2)*1024\n\t.endif\n\t"
      ".if %9 > 4\n\tglobal_load_lds_dwordx4 %4, off offset:(4-%9/2)*1024\n\t.endif\n\t"
      ".if %9 > 5\n\tglobal_load_lds_dwordx4 %5, off offset:(5-%9/2)*1024\n\t.endif\n\t"
      ".if %9 > 6\n\tglobal_load_lds_dwordx4 %6, off offset:(6-%9/2)*1024\n\t.endif\n\t"
      ".if %9 > 7\n\tglobal_load_lds_dwordx4 %7, off offset:(7-%9/2)*1024\n\t.endif"
      :
      : "v"(g[0]), "v"(g[1]), "v"(g[2]), "v"(g[3]), "v"(g[4]), "v"(g[5]), "v"(g[6]), "v"(g[7]), "s"(m0v), "n"(N)
      : "memory");
}

// The same burst for loads whose lanes all read from one wave-uniform base: address = base (SGPR pair)
// + off[i] (unsigned 32-bit, per lane) + immediate.  No 64-bit address arithmetic and one VGPR per load.
// The caller passes off[i] = byte offset from base - (i - N/2) KiB, which must not be negative.  ONCE: bytes that nobody reads
// again (nontemporal: they leave the caches what they hold).
template <int N, bool ONCE = false>
AE_DEV void ae_load_lds16_burst_base(const void* base, const unsigned* off, ae_lds_u8* lds_mid) {
  static_assert(N >= 1 && N <= 8, "the 13-bit signed immediate offset reaches -4 KiB .. +3 KiB");
  const unsigned m0v = __builtin_amdgcn_readfirstlane((unsigned)(unsigned long)lds_mid);
  // the base must sit in scalar registers even where the compiler cannot prove it wave uniform
  const unsigned long bv = (unsigned long)base;
  // (readfirstlane returns a signed int: go through unsigned, or the low half sign-extends into the high)
  const unsigned b_hi = (unsigned)__builtin_amdgcn_readfirstlane((unsigned)(bv >> 32));
  const unsigned b_lo = (unsigned)__builtin_amdgcn_readfirstlane((unsigned)bv);
  const unsigned long ub = ((unsigned long)b_hi << 32) | (unsigned long)b_lo;
  if constexpr (ONCE)
    asm volatile(
        "s_mov_b32 m0, %8\n\ts_nop 0\n\t"
        "global_load_lds_dwordx4 %0, %10 offset:(0-%9/2)*1024 nt\n\t"
        ".if %9 > 1\n\tglobal_load_lds_dwordx4 %1, %10 offset:(1-%9/2)*1024 nt\n\t.endif\n\t"
        ".if %9 > 2\n\tglobal_load_lds_dwordx4 %2, %10 offset:(2-%9/2)*1024 nt\n\t.endif\n\t"
        ".if %9 > 3\n\tglobal_load_lds_dwordx4 %3, %10 offset:(3-%9/2)*1024 nt\n\t.endif\n\t"
        ".if %9 > 4\n\tglobal_load_lds_dwordx4 %4, %10 offset:(4-%9/2)*1024 nt\n\t.endif\n\t"
        ".if %9 > 5\n\tglobal_load_lds_dwordx4 %5, %10 offset:(5-%9/2)*1024 nt\n\t.endif\n\t"
        ".if %9 > 6\n\tglobal_load_lds_dwordx4 %6, %10 offset:(6-%9/2)*1024 nt\n\t.endif\n\t"
        ".if %9 > 7\n\tglobal_load_lds_dwordx4 %7, %10 offset:(7-%9/2)*1024 nt\n\t.endif"
        :
        : "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "v"(off[4]), "v"(off[5]), "v"(off[6]), "v"(off[7]),
          "s"(m0v), "n"(N), "s"(ub)
        : "memory");
  else
    asm volatile(
        "s_mov_b32 m0, %8\n\ts_nop 0\n\t"
        "global_load_lds_dwordx4 %0, %10 offset:(0-%9/2)*1024\n\t"
        ".if %9 > 1\n\tglobal_load_lds_dwordx4 %1, %10 offset:(1-%9/2)*1024\n\t.endif\n\t"
        ".if %9 > 2\n\tglobal_load_lds_dwordx4 %2, %10 offset:(2-%9/2)*1024\n\t.endif\n\t"
        ".if %9 > 3\n\tglobal_load_lds_dwordx4 %3, %10 offset:(3-%9/2)*1024\n\t.endif\n\t"
        ".if %9 > 4\n\tglobal_load_lds_dwordx4 %4, %10 offset:(4-%9/2)*1024\n\t.endif\n\t"
        ".if %9 > 5\n\tglobal_load_lds_dwordx4 %5, %10 offset:(5-%9/2)*1024\n\t.endif\n\t"
        ".if %9 > 6\n\tglobal_load_lds_dwordx4 %6, %10 offset:(6-%9/2)*1024\n\t.endif\n\t"
        ".if %9 > 7\n\tglobal_load_lds_dwordx4 %7, %10 offset:(7-%9/2)*1024\n\t.endif"
        :
        : "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "v"(off[4]), "v"(off[5]), "v"(off[6]), "v"(off[7]),
          "s"(m0v), "n"(N), "s"(ub)
        : "memory");
}

// The same burst through a buffer resource whose range ends with the last row: 16-byte chunks past it arrive as zeros.
// A tile that the end of the sequence cuts then needs no per-lane clamping (in the loop: eight address selects a tensor
// and tile, and the registers for them), and its missing rows are zeros.  Loads 4n .. 4n + 3 go out behind one write of
// M0; the 12-bit immediate moves the LDS and the global address, so off[i] = byte offset in the tile + 4096 -
// (i % 4) KiB from a base that is passed 4 KiB low (offsets and range stay positive), `bytes` = the tile's valid bytes.
template <int N>
AE_DEV void ae_load_lds16_burst_rows(const void* base, unsigned bytes, const unsigned* off, ae_lds_u8* lds_first) {
  static_assert(N >= 1 && N <= 8, "at most two bursts of four");
  const unsigned long bv = (unsigned long)base;
  const ae_u32x4 rsrc = {(unsigned)__builtin_amdgcn_readfirstlane((unsigned)bv),
                         (unsigned)__builtin_amdgcn_readfirstlane((unsigned)(bv >> 32)) & 0xffffu,
                         (unsigned)__builtin_amdgcn_readfirstlane(bytes + 4096u), 0x00020000u};
  const unsigned m0a = __builtin_amdgcn_readfirstlane((unsigned)(unsigned long)lds_first);
  asm volatile(
      "s_mov_b32 m0, %4\n\ts_nop 0\n\t"
      "buffer_load_dwordx4 %0, %5, 0 offen lds\n\t"
      ".if %6 > 1\n\tbuffer_load_dwordx4 %1, %5, 0 offen offset:1024 lds\n\t.endif\n\t"
      ".if %6 > 2\n\tbuffer_load_dwordx4 %2, %5, 0 offen offset:2048 lds\n\t.endif\n\t"
      ".if %6 > 3\n\tbuffer_load_dwordx4 %3, %5, 0 offen offset:3072 lds\n\t.endif"
      :
      : "v"(off[0]), "v"(off[N > 1 ? 1 : 0]), "v"(off[N > 2 ? 2 : 0]), "v"(off[N > 3 ? 3 : 0]), "s"(m0a), "s"(rsrc), "n"(N)
      : "memory");
  if constexpr (N > 4) ae_load_lds16_burst_rows<N - 4>(base, bytes, off + 4, lds_first + 4096);
}

// ---- transcendentals ------------------------------------------------------------------
AE_DEV float ae_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
AE_DEV float ae_exp(float x) { return __builtin_amdgcn_exp2f(x * AE_LOG2E); }
AE_DEV float ae_log2(float x) { return __builtin_amdgcn_logf(x); }
AE_DEV float ae_log(float x) { return __builtin_amdgcn_logf(x) * AE_LN2; }
AE_DEV float ae_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
// tanh(x) = 1 - 2 / (exp(2x) + 1); saturates cleanly at +-1 for large |x|.
AE_DEV float ae_tanh(float x) {
  float e = __builtin_amdgcn_exp2f(x * (2.0f * AE_LOG2E));
  return 1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f);
}
AE_DEV float ae_abs(float x) { return __builtin_fabsf(x); }
AE_DEV float ae_max(float a, float b) { return __builtin_fmaxf(a, b); }

// ---- exchange between the lanes that share one query row -----------------------------------
// AE_LAYOUT 0 (prefill, 32x32x16 MFMA, S^T accumulators): a row lives in lanes l and l^32.
//   permlane32_swap with both operands equal returns (value of the low half, value of the
//   high half) in every lane of the pair.
// AE_LAYOUT 1 (decode, 16x16x32 MFMA): a row (one query head) lives in lanes l, l^16, l^32, l^48.
#ifndef AE_LAYOUT
#define AE_LAYOUT 0
#endif
AE_DEV float ae_swap32_lo_hi(float v, float& hi) {
  unsigned u = __builtin_bit_cast(unsigned, v);
  auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  hi = __builtin_bit_cast(float, (unsigned)r[1]);
  return __builtin_bit_cast(float, (unsigned)r[0]);
}
// the values of the even and of the odd 16-lane row of a lane's row pair (v_permlane16_swap with both operands
// equal): an exchange inside the VALU, where ds_bpermute goes through the LDS pipeline and back
AE_DEV float ae_swap16_even_odd(float v, float& odd) {
  unsigned u = __builtin_bit_cast(unsigned, v);
  auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  odd = __builtin_bit_cast(float, (unsigned)r[1]);
  return __builtin_bit_cast(float, (unsigned)r[0]);
}
AE_DEV float ae_group_max(float v) {
#if AE_LAYOUT == 1
  {
    float od;
    const float ev = ae_swap16_even_odd(v, od);
    v = __builtin_fmaxf(ev, od);
  }
#endif
  float hi;
  float lo = ae_swap32_lo_hi(v, hi);
  return __builtin_fmaxf(lo, hi);
}
AE_DEV float ae_group_sum(float v) {
#if AE_LAYOUT == 1
  {
    float od;
    const float ev = ae_swap16_even_odd(v, od);
    v = ev + od;
  }
#endif
  float hi;
  float lo = ae_swap32_lo_hi(v, hi);
  return lo + hi;
}

// ---- row reductions over the lane's slice of a score row + the lanes sharing the row --------
// (ReduceMax / ReduceSum / ReduceAbsSum over dim=1 of the [block_M, block_N] tile,
//  core/codegen/tl_gen.py:9-21.)
template <int N>
AE_DEV float ae_lane_max(const float (&s)[N]) {
  float m = s[0];
#pragma unroll
  for (int e = 1; e < N; e++) m = __builtin_fmaxf(m, s[e]);
  return m;
}
template <int N>
AE_DEV float ae_row_max(const float (&s)[N]) {
  return ae_group_max(ae_lane_max<N>(s));
}
template <int N>
AE_DEV float ae_lane_sum(const float (&s)[N]) {
  // four independent chains keep the adds off one dependency path
  float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
#pragma unroll
  for (int e = 0; e + 3 < N; e += 4) {
    a0 += s[e];
    a1 += s[e + 1];
    a2 += s[e + 2];
    a3 += s[e + 3];
  }
#pragma unroll
  for (int e = N & ~3; e < N; e++) a0 += s[e];
  return (a0 + a1) + (a2 + a3);
}
template <int N>
AE_DEV float ae_row_sum(const float (&s)[N]) {
  return ae_group_sum(ae_lane_sum<N>(s));
}
template <int N>
AE_DEV float ae_row_abssum(const float (&s)[N]) {
  float a0 = 0.f, a1 = 0.f;
#pragma unroll
  for (int e = 0; e + 1 < N; e += 2) {
    a0 += __builtin_fabsf(s[e]);
    a1 += __builtin_fabsf(s[e + 1]);
  }
#pragma unroll
  for (int e = N & ~1; e < N; e++) a0 += __builtin_fabsf(s[e]);
  return ae_group_sum(a0 + a1);
}

// ---- reductions over the split axis (ColReduce*, used by OnlineFunc.combine) -----------------
template <int N>
AE_DEV float ae_arr_max(const float (&s)[N]) {
  float m = s[0];
#pragma unroll
  for (int e = 1; e < N; e++) m = __builtin_fmaxf(m, s[e]);
  return m;
}
template <int N>
AE_DEV float ae_arr_sum(const float (&s)[N]) {
  float a = 0.f;
#pragma unroll
  for (int e = 0; e < N; e++) a += s[e];
  return a;
}
template <int N>
AE_DEV float ae_arr_abssum(const float (&s)[N]) {
  float a = 0.f;
#pragma unroll
  for (int e = 0; e < N; e++) a += __builtin_fabsf(s[e]);
  return a;
}

// Per-row context handed to the functors.
struct ae_ctx {
  int b;        // batch index
  int h;        // query head index
  int q_idx;    // absolute query position of this lane's row
  int kv_base;  // absolute kv position of element 0 of the lane's slice in the current tile
};

// kv offset (relative to ae_ctx::kv_base) of element e of a lane's slice of a score row.
// AE_LAYOUT 0: the slice is NB accumulator blocks of 16; block nb covers kv 32*nb .. 32*nb+31 and
//   register r of half-wave hf holds kv 8*(r/4) + 4*hf + r%4 (4*hf is folded into kv_base).
// AE_LAYOUT 1: blocks of 4; block rb covers kv 16*rb .. 16*rb+15 and register r of lane group g
//   holds kv 4*g + r (4*g is folded into kv_base).
#if AE_LAYOUT == 1
AE_DEV constexpr int ae_kv_off(int e) { return (e >> 2) * 16 + (e & 3); }
#else
AE_DEV constexpr int ae_kv_off(int e) { return (e >> 4) * 32 + ((e & 15) >> 2) * 8 + (e & 3); }
#endif

// ---- paged launches whose splits follow the entries' lengths (ae_attn_params.tail_slots; batches of at most 64) ------------
// inclusive scan over the wave's lanes, all of them active: sums, or maxima of numbers >= 0
template <bool MAX>
AE_DEV int ae_wave_scan(int x) {
  auto step = [&](int y) AE_LAMBDA { x = MAX ? (x > y ? x : y) : x + y; };
  step(__builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false));      // row_shr 1, 2, 4, 8
  step(__builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false));
  step(__builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false));
  step(__builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false));
  step(__builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false));      // row_bcast 15, 31
  step(__builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false));
  return x;
}
// The kv axes of all entries cut into splits of `tiles` kv tiles, at most a sixteenth above the least with which p.tail_slots workgroups
// a head tile suffice and no entry has more than p.num_splits: lane b's entry has `mine` of them (one at least), the entries up to it `upto`.
// Equal spans of the table, which the host can plan, leave the workgroups without keys whose spans lie behind an entry's end, and the
// launch takes as long as the longest entry's.  Every wave works this out from the lengths (0.2 us, and they are one trip to
// memory that the first requests wait for: 0.2 to 0.8 us of a call).  us, equal spans -> so, entries spread evenly up to the table's width |
// all of that width: B64 H128 4096 85.7 -> 61.9 | 130.8 -> 93.1, B21 H64 2624 23.7 -> 20.9 | 40.6 -> 26.8.  Where equal spans are one round of
// the CUs, full tables are the slower for it (B8 H128 2048 18.7 -> 17.4 | 19.9 -> 20.2).  Which calls take it: MLADecodeOp._splits_by_length.
struct ae_paged_splits { int tiles, mine, upto; };
#define AE_LEAST_TILES 4      // (a split's start and end, and its partial result, take as long as four trips)
AE_DEV ae_paged_splits ae_split_by_length(const ae_attn_params& p, int lane, int entry_tiles) {
  ae_paged_splits s;
  const bool there = lane < p.batch;
  entry_tiles = there ? entry_tiles : 0;
  const int total = __builtin_amdgcn_readlane(ae_wave_scan<false>(entry_tiles), 63);
  int rest;           // (an entry has at most 2^19 tiles, and there are at most p.tail_slots entries: the quotient is no more than that)
  s.tiles = ae_divide_small(total + p.tail_slots - 1, p.tail_slots, rest);
  s.tiles = s.tiles > AE_LEAST_TILES ? s.tiles : AE_LEAST_TILES;
  for (;;) {            // (ends: with s.tiles at the longest entry's every entry has one split, and there are at most p.tail_slots entries)
    const int a = entry_tiles + s.tiles - 1;
    int n = (int)((float)a * __builtin_amdgcn_rcpf((float)s.tiles));       // off by at most one below 2^22
    n -= n * s.tiles > a ? 1 : 0;
    n += a - n * s.tiles >= s.tiles ? 1 : 0;
    s.mine = there ? (n > 1 ? n : 1) : 0;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(s.mine > p.num_splits) != 0, 0)) {      // (one entry far longer than the others)
      const int most = __builtin_amdgcn_readlane(ae_wave_scan<true>(entry_tiles), 63);
      s.tiles = ae_divide_small(most + p.num_splits - 1, p.num_splits, rest);
      continue;
    }
    s.upto = ae_wave_scan<false>(s.mine);
    if (__builtin_amdgcn_readlane(s.upto, 63) <= p.tail_slots) return s;
    s.tiles += s.tiles >> 4 > 1 ? s.tiles >> 4 : 1;
  }
}

#endif  // AE_DEVICE_H
