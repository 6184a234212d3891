// bkv_mfma16.h - building blocks on the fp16 and fp32 matrix cores shared by the prefill and
// short-context kernels: exact fp16 operands of q8_0 bytes, the two-digit q16 operands of the q8_0
// scores, the serial fp16 score chain, p16's quotient, and the LDS-only barrier.
#pragma once

#include "bkv_common.h"
#include "bkv_q8dot.h"

namespace bkv {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef short v4s_t __attribute__((ext_vector_type(4)));
typedef short v8s_t __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f4 mfma16(h8 a, h8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ h2 as_h2(uint32_t w) { return __builtin_bit_cast(h2, w); }
__device__ __forceinline__ uint32_t as_u(h2 v) { return __builtin_bit_cast(uint32_t, v); }

// two signed bytes of w (already biased by 0x80 per byte), selected by SEL, as an exact fp16 pair:
// 0x64XX is the fp16 number 1024 + XX, so subtracting 1152 leaves the signed byte value.
template <uint32_t SEL>
__device__ __forceinline__ h2 bytes_h2(uint32_t wb) {
  const h2 x = as_h2(__builtin_amdgcn_perm(0x64646464u, wb, SEL));
  return x - h2{(_Float16)1152.0f, (_Float16)1152.0f};
}

// e / s correctly rounded to fp32, from rs = fp32(1/s) correctly rounded, without a division:
// q0 = e*rs is within 1.5 ulps of e/s; one correction q1 = q0 + (e - s*q0)*rs (the remainder exact
// by fma) brings it within one ulp, and a second is then the correctly rounded quotient (Markstein's
// theorem: y within half an ulp of 1/s, q within one ulp of e/s, r = e - s*q exact => RN(q + r*y)
// = RN(e/s)). Valid for 0 <= e <= s, s >= 1 (a softmax sum includes the maximum's e = 1): the
// remainders stay normal while the quotient is above 2^-60, and below that the quotient rounds to
// an fp16 zero whatever its last bits.
__device__ __forceinline__ float div_by_sum(float e, float s, float rs) {
  const float q0 = e * rs;
  const float q1 = __builtin_fmaf(__builtin_fmaf(-s, q0, e), rs, q0);
  float q2 = __builtin_fmaf(__builtin_fmaf(-s, q1, e), rs, q1);
  // the fp32 result itself: a conversion to fp16 of the fma would otherwise be folded into one
  // mixed-precision fma rounding once, straight to fp16 (a different result at fp16 ties)
  asm volatile("" : "+v"(q2));
  return q2;
}

// exact fp16 split of s*b: hi = f16(s*b) (rounded fp16 product), lo = the product's rounding error
__device__ __forceinline__ void split_prod(h2 b, h2 s, h2 &hi, h2 &lo) {
  hi = b * s;
  lo = __builtin_elementwise_fma(b, s, -hi);
}

// ---------------------------------------------------------------- V tiles outside the plain products
// The PV kernels multiply p16 with fp16 operands of V: the values themselves (fp16 V), or d * b split in
// two (q8_0 V). Two kinds of tile need more than that, and take pv_tile_careful instead:
//  * a q8_0 scale of 512 or more (scale_big), whose products leave fp16: such a key enters a second pair
//    of operands as (d * 2^-8) * b against p16 * 2^8, both exact (d is at least 2 there, p16 at most 1);
//  * keys that some of the rows do not see (later queries' keys, padding) beside a value that is Inf or
//    NaN: p = 0 does not take them out, as 0 * Inf is NaN. The rows of one query at a time are computed with
//    the keys past that query's last one zeroed in the V operand, and the other rows' results dropped.
// A tile of either kind costs up to 2 x 4 times the MFMAs; ordinary values never have one. (us, with ordinary
// scales and with every scale past 512: a decode of 300 keys 12.8 / 19.0, 6 queries onto 300 keys 16.6 / 26.9,
// 6 onto 3000 44.1 / 58.8, 512 onto 8192 333 / 430.)

// bits 14 and 30: the low and high fp16 of w is 512 or more in magnitude, Inf or NaN
__device__ __forceinline__ uint32_t scale_big(uint32_t w) { return w & (w << 1) & 0x40004000u; }
// bits 15 and 31: the low and high fp16 of w is Inf or NaN
__device__ __forceinline__ uint32_t non_finite(uint32_t w) { return ((w & 0x7C007C00u) + 0x04000400u) & 0x80008000u; }
// 0xFFFF in the halves whose flag (bit N of each) is set
template <int N>
__device__ __forceinline__ uint32_t half_mask(uint32_t flags) { return (flags >> N) * 0xFFFFu; }

// One 64-key tile (first key key0) against NTR tiles of 16 rows: lane l's accumulators o[mt][nt] hold row
// 16 nt + l % 16, i.e. the chunk's query 4 nt + (l % 16) / 4, whose last key is lim0 + 4 nt + (l % 16) / 4.
// l: the accumulators of the products' small parts (o itself will do).
// masked: some row does not see all of the tile's keys (NQ queries per row tile). ops(ks, mt, x, s): the V
// operand of the lane's keys key0 + 32 ks + 8 (l / 16) .. + 7 in pairs: fp16 V x; q8_0 V the bytes x and
// scales s as fp16. rows(ks, nt): their p16.
template <int VF, int NTR, int NQ, typename OPS, typename ROWS>
__device__ __forceinline__ void pv_tile_careful(f4 (&o)[2][NTR], f4 (&l)[2][NTR], int key0, int lim0, bool masked, const OPS &ops, const ROWS &rows) {
  constexpr int NA = VF ? 4 : 1;                   // the products' small parts, then the large ones
  const int lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4;
#pragma unroll 1
  for (int ks = 0; ks < 2; ++ks) {
    const int k0 = key0 + 32 * ks + 8 * lq;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      uint32_t x[4], s[4], a[NA][4];
      ops(ks, mt, x, s);
#pragma unroll
      for (int pp = 0; pp < 4; ++pp) {
        if constexpr (VF) {
          const uint32_t big = half_mask<14>(scale_big(s[pp]));
          h2 hi, lo;
          split_prod(as_h2(x[pp]), as_h2(s[pp] & ~big), hi, lo);
          a[0][pp] = as_u(lo);
          a[2][pp] = as_u(hi);
          split_prod(as_h2(x[pp]), as_h2(s[pp] & big) * h2{(_Float16)0x1p-8f, (_Float16)0x1p-8f}, hi, lo);
          a[1][pp] = as_u(lo) & ~half_mask<15>(non_finite(as_u(hi)));   // (Inf - Inf: the Inf is in hi)
          a[3][pp] = as_u(hi);
        } else {
          a[0][pp] = x[pp];
        }
      }
#pragma unroll 1
      for (int qi = 0; qi < (masked ? NQ : 1); ++qi) {
        const bool mine = !masked || (lr >> 2) == qi;
        asm volatile("" ::: "memory");             // (the rows' p16 read again for each query: their registers)
#pragma unroll
        for (int nt = 0; nt < NTR; ++nt) {
          const int seen = masked ? lim0 + 4 * nt + qi - k0 : 7;             // the lane's keys 0 .. seen
          uint32_t m[4];
#pragma unroll
          for (int pp = 0; pp < 4; ++pp) m[pp] = (2 * pp <= seen ? 0xFFFFu : 0u) | (2 * pp + 1 <= seen ? 0xFFFF0000u : 0u);
          const _Float16 f = (_Float16)256.0f;
          h8 p[2];                                 // p16 and p16 * 2^8
          p[0] = rows(ks, nt);
          p[1] = p[0] * h8{f, f, f, f, f, f, f, f};
#pragma unroll
          for (int j = 0; j < (VF ? 2 : 1); ++j) { // (the plain products' order)
            f4 &acc = VF && j == 0 ? l[mt][nt] : o[mt][nt];
            f4 t = acc;
#pragma unroll
            for (int i = 0; i < (VF ? 2 : 1); ++i) {
              const uint32_t (&b)[4] = a[2 * j + i];
              t = mfma16(__builtin_bit_cast(h8, make_uint4(b[0] & m[0], b[1] & m[1], b[2] & m[2], b[3] & m[3])), p[i], t);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = mine ? t[i] : acc[i];
          }
        }
      }
    }
  }
}

// Workgroup barrier for LDS traffic only: every wave's LDS operations have completed, while its
// global loads (prefetches a step or more ahead) stay in flight. __syncthreads() also releases
// global memory, i.e. waits for every outstanding load and store of the wave first, which would
// void those prefetches. Used where the waves exchange data through LDS alone.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ---------------------------------------------------------------- q8_0 K scores on the matrix cores
// The contract's inner sum (bkv_q8dot.h) is the fp32 rounding of the exact sum of q16 * int8 over a
// block. fp16 MFMAs give it with two digits per q16, q = hi + lo: hi a multiple of u and lo a multiple
// of t, where u is the smallest power of two with sum |hi| * 128 <= 2^24 u in every block of the row, and
// sum |lo| * 128 <= 2^24 t. All products of a digit with bytes in [-128, 127] and all their partial sums
// are then multiples of the digit's unit below 2^24 units: the MFMA's fp32 sums are exact in any
// order, and fp32(hi sum + lo sum) is one fma with one rounding (lo is kept scaled by 2^8): one VALU
// instruction per block and score, where int8 digits need two shifted adds, two conversions, an fma in
// fp64 and its rounding. The row is scaled by a power of two so that u = 2^-2: hi <= 2^15, lo * 2^8 <= 2^5
// in units above 2^-14, all fp16 normals; hi has at most 11 significant bits (a q16 of 2^10 u or more is
// itself a multiple of u), lo at most 11 (it is q16 or a remainder of it).
// A block whose lo is no multiple of such a t in some row (a q16 about 2^-16 of the row's largest or
// less: one of a hundred rows of normal values has one) gets a third digit: lo a multiple of 2^-13 u,
// lo2 = the rest, a multiple of 2^-26 u, kept scaled by 2^14. It costs a third MFMA, and its three sums
// are combined in fp64 (below 2^53 units: exact) and rounded once. Rows that need more, or hold Inf / NaN,
// take the fp64 VALU path.
constexpr int kQ8fUnit = 2 * 8 * 64;               // 16-byte operands per unit: [pair j][block][lane]

// Cooperative (256 threads, tid their index): the A operands of a unit's q rows in dig [pair][block][lane] (pair j: rows 4 i + 2 (h % 2) + digit for heads h = 2 j,
// 2 j + 1 of query i) and lo2 [block][lane] (rows 4 i + h); lane l of an operand holds row l % 16, dims
// 8 (l/16) .. + 7 of the block. ex[row 4 i + h]: the score's power of two. *flags: bit b set when block b
// of any row has a third digit; *wide when the rows need the fp64 path. Both zeroed by the caller.
// raw: what q8f_fetch loaded (apart, so that a caller can have other loads queue behind it).
struct Q8fRaw { f4 v[4]; };                        // row tid / 16 (query, head), dims 16 (tid % 16) .. + 15
template <typename ROWS>
__device__ __forceinline__ void q8f_fetch(int tid, const ROWS &rows, int qs, Q8fRaw &raw) {   // rows(i): query i's 4 head rows
  const float *src = rows(tid >> 6) + (size_t)((tid >> 4) & 3) * qs + 16 * (tid & 15);
#pragma unroll
  for (int i = 0; i < 4; ++i) raw.v[i] = *reinterpret_cast<const f4 *>(src + 4 * i);
}
__device__ __forceinline__ void q8f_digits(int tid, const Q8fRaw &raw, uint4 *dig, uint4 *lo2, float *ex, unsigned *flags,
                                           unsigned *wide) {
  const int r = tid >> 4, p = tid & 15, qi = r >> 2, h = r & 3;
  float x[16], s = 0.0f;
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f4 t = raw.v[i];
    x[4 * i] = round_f16(t.x); x[4 * i + 1] = round_f16(t.y);
    x[4 * i + 2] = round_f16(t.z); x[4 * i + 3] = round_f16(t.w);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    bad = bad || !(fabsf(x[i]) <= 65504.0f);
    s += fabsf(x[i]);
  }
  s += dpp<0xB1>(s);                               // the block's (two lanes hold one)
  s = row16_max(s);                                // the row's largest
  // S = s below 2^(E+1) (below 0.999 of it, for s's rounding and the u/2 that rounding adds to each hi):
  // u = 2^(E-16); scaled so that u = 2^-2
  const uint32_t sb = __float_as_uint(s);
  const int E = s > 0.0f ? (int)(sb >> 23) - 127 + ((sb & 0x7FFFFFu) > 0x7FBFFFu ? 1 : 0) : 14;
  bad = bad || E > 100;                            // (Inf / NaN rows: any finite scale)
  const float up = bad ? 1.0f : __uint_as_float((uint32_t)(127 + 14 - E) << 23);
  float lr[16], L = 0.0f;
  h8 d0[2], d1[2], d2[2];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float y = x[i] * up;                     // exact
    const float hi = __builtin_rintf(y * 4.0f) * 0.25f;
    lr[i] = y - hi;                                // exact, at most 2^-3
    L += fabsf(lr[i]);
    d0[i >> 3][i & 7] = (_Float16)hi;
  }
  L += dpp<0xB1>(L);
  // t = 2^(exponent of L + 1 - 17), at least 2^-22: L * 128 < 2^24 t (L's fp32 rounding is far below the
  // factor of up to 2 that the exponent leaves, except where L is within 2^-18 of a power of two: + 1)
  const uint32_t lb = __float_as_uint(L) + 64u;
  const float ti = __uint_as_float((uint32_t)(254 - max((int)(lb >> 23) + 1 - 17, 127 - 22)) << 23);   // 1 / t
  bool fine = true;
#pragma unroll
  for (int i = 0; i < 16; ++i) fine = fine && __builtin_rintf(lr[i] * ti) == lr[i] * ti;
  const bool third = !(fine && dpp<0xB1>(fine ? 1.0f : 0.0f) == 1.0f);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float lo = third ? __builtin_rintf(lr[i] * 32768.0f) * 0x1p-15f : lr[i];
    const float l2 = (lr[i] - lo) * 16384.0f;      // exact, at most 2^-2
    bad = bad || __builtin_rintf(l2 * 16384.0f) != l2 * 16384.0f;
    d1[i >> 3][i & 7] = (_Float16)(lo * 256.0f);
    d2[i >> 3][i & 7] = (_Float16)l2;
  }
  const int b = p >> 1;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int lq = 2 * (p & 1) + k, l = 16 * lq + 4 * qi + 2 * (h & 1);
    uint4 *o = dig + ((h >> 1) * 8 + b) * 64;
    o[l] = __builtin_bit_cast(uint4, d0[k]);
    o[l + 1] = __builtin_bit_cast(uint4, d1[k]);
    lo2[b * 64 + 16 * lq + r] = __builtin_bit_cast(uint4, d2[k]);
  }
  if (p == 0) ex[r] = 1.0f / up;
  if (third) atomicOr(flags, 1u << b);
  if (bad) atomicOr(wide, 1u);
}

typedef float fv16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ fv16 mfma_k1(float a, float b, fv16 c) {
  return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t word_of(const uint4 &v, int i) {
  return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
}

}  // namespace bkv
