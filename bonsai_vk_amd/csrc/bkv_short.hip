// bkv_short.hip - attention over at most kShortKeys keys in one workgroup per KV group and query
// (decode) or per KV group and 4 queries (prefill chunks): no exchange between workgroups at all.
//
// The stream kernel takes 18 us however short the context, nearly all of it its three exchanges
// between workgroups; the chunk pipeline takes 40-48 us in four launches. Here the whole row fits one CU:
// the scores of up to 16 rows x 512 keys stay in LDS (33 KiB), e replaces them, one lane per row adds
// e in key order (the reference's serial fp32 sum, attn_vk.h:175-189), p16 = f16(e / sum) goes to LDS and
// the PV runs on the matrix cores from V tiles that direct-to-LDS loads brought in behind the scores.
// What bounds it: a chain of latencies (K rows, scores, exps, the serial sum at about 5 ns per key, V
// tiles); past 384, 448 or 512 keys, by format and layout, a decode is faster where the stream or resident
// kernel spreads the keys wider (short_decode_keys). Chunks take it to kShortKeys (short_chunk).
// Scores, e, sums and p16 are bit-identical to the other kernels'; the PV sum's order differs. Its error
// given p16 (2-norm, q8_0 V) is 6.6e-8 at 64 keys, 7.7e-8 at 300, 8.5e-8 at 440 (the stream kernel's 6.9e-8,
// 8.5e-8, 8.6e-8; one fp32 chain over all products 8.8e-8, 1.7e-7, 2.0e-7).
#include <type_traits>

#include "bkv_device.h"
#include "bkv_exp.h"
#include "bkv_internal.h"
#include "bkv_mfma16.h"
#include "bkv_pv8.h"

namespace bkv {

constexpr int kShNT = 512;                         // 8 waves
constexpr int kShKS = kShortKeys + 4;              // floats per score row (rows 4 banks apart)
constexpr int kShPS = 2 * kShortKeys + 16;         // bytes per p16 row

__device__ __forceinline__ uint32_t half_of(const uint4 &v, int i) {   // 16-bit element i of 8
  const uint32_t w = i < 2 ? v.x : i < 4 ? v.y : i < 6 ? v.z : v.w;
  return (i & 1) ? (w >> 16) : (w & 0xFFFFu);
}

// NR: rows of the workgroup, 4 (one query x 4 heads) or 16 (4 queries x 4 heads)
template <int KF, int VF, int NR, bool PG>
__global__ __launch_bounds__(kShNT, 1) void short_kernel(ShortArgs a) {
  constexpr int NQ = NR / kGqa, VB = VF ? 16384 : 32768, ND = VF ? 2 : 4;
  constexpr int NB = VF ? (NR == 4 ? 7 : 4) : 3;   // V tiles in LDS
  const int g = blockIdx.x % a.nkv, q0 = NQ * (blockIdx.x / a.nkv);
  const int nqv = min(NQ, a.n_q - q0);
  const int kend = (int)a.pos0 + q0 + nqv;         // keys 0 .. kend - 1, at most kShortKeys
  const int nt = (kend + 63) >> 6;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  const bool append = NR == 4 && a.ap.k != nullptr;
  constexpr int KRB = row_bytes(KF ? BKV_Q8_0 : BKV_F16), VRB = row_bytes(VF ? BKV_Q8_0 : BKV_F16);

  __shared__ __attribute__((aligned(1024))) char s_v[NB][VB];
  __shared__ __attribute__((aligned(16))) char s_p[16 * kShPS];   // first the q16 operands
  __shared__ __attribute__((aligned(16))) float s_sc[NR][kShKS];
  __shared__ uint4 s_vs[VF ? kShortKeys : 1];      // the keys' V scale rows
  __shared__ uint4 s_lo2[KF && NR == 16 ? 8 * 64 : 1];
  __shared__ uint4 s_row[2][33];                   // the appended K and V row: data, then scales
  __shared__ __attribute__((aligned(16))) float s_new[2][kHd], s_q4[NR == 4 ? kGqa : 1][kHd];
  __shared__ double s_t2[32];
  __shared__ __attribute__((aligned(16))) float s_gate[NR == 4 ? NR * kHd : 4];  // 1 / (1 + exp(-gate))
  __shared__ float s_ex[16], s_red[8][NR], s_sum[NR];
  __shared__ int s_lt[kGqa];
  __shared__ unsigned s_flags, s_wide, s_big;      // (s_big: a V scale past the plain products)
  if (tid == 0) { s_flags = 0u; s_wide = 0u; s_big = 0u; }
  if (tid < 32) s_t2[tid] = kExp2Tab[tid];
  static_assert(16 * kShPS >= kQ8fUnit * 16 && 16 * kShPS >= kHd * 16 * 4 && 16 * kShPS >= kLimBytes, "q16 operands in s_p");
  lds_barrier();

  auto qrows = [&](int i) { return a.q + ((size_t)min(q0 + i, a.n_q - 1) * a.nh + g * kGqa) * a.qs; };
  auto krow = [&](int key) { return slot_t<PG>(a.L, min(key, kend - 1)) * a.nkv + g; };
  float mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  // the appended token (wave 7; lanes 0..31 K, 32..63 V): its rows are requested in front of the cached
  // ones and quantised once, into the cache and into s_row for this workgroup (whose loads of that row may
  // return what was there before)
  f4 nr0 = {0.f, 0.f, 0.f, 0.f}, nr1 = nr0;
  if (append && w == 7) {
    const f4 *src = reinterpret_cast<const f4 *>((lane < 32 ? a.ap.k : a.ap.v) + (size_t)g * kHd) + 2 * (lane & 31);
    nr0 = src[0];
    nr1 = src[1];
  }
  __builtin_amdgcn_sched_barrier(0);
  auto append_new = [&]() {
    reinterpret_cast<f4 *>(&s_new[lane >> 5][0])[2 * (lane & 31)] = nr0;
    reinterpret_cast<f4 *>(&s_new[lane >> 5][0])[2 * (lane & 31) + 1] = nr1;
    __builtin_amdgcn_wave_barrier();
    const int64_t slot = slot_of(a.ap.L, a.ap.pos);
    if (lane < 32) {
      const PackedRow r = pack_row<KF, false>(s_new[0], lane);
      store_row<KF>(r, const_cast<uint8_t *>(a.ap.L.kd) + (slot * a.nkv + g) * KRB,
                    KF ? const_cast<uint8_t *>(a.ap.L.ks) + (slot * a.nkv + g) * kScaleRowBytes : nullptr, lane);
      store_row<KF>(r, reinterpret_cast<uint8_t *>(&s_row[0][0]), reinterpret_cast<uint8_t *>(&s_row[0][16]), lane);
    } else {
      const PackedRow r = pack_row<VF, false>(s_new[1], lane - 32);
      store_row<VF>(r, const_cast<uint8_t *>(a.ap.L.vd) + (slot * a.nkv + g) * VRB,
                    VF ? const_cast<uint8_t *>(a.ap.L.vs) + (slot * a.nkv + g) * kScaleRowBytes : nullptr, lane - 32);
      store_row<VF>(r, reinterpret_cast<uint8_t *>(&s_row[1][0]), reinterpret_cast<uint8_t *>(&s_row[1][16]), lane - 32);
    }
  };

  // ---------------------------------------------------------------- scores
  if constexpr (KF) {
    // wave w: key groups w, w + 8, .. (16 keys each); lane: key 16 kg + lr, bytes 64 j + 16 lq .. +
    // 15 (half the loads of 8-byte pieces; the halves then change places between lanes, see below). The
    // number of rounds is a constant in each copy: behind conditional loads the wait for the q rows would
    // be one for every K row.
    auto scores = [&](auto rounds) {
      constexpr int NC = rounds.value;
      struct KG { u32x4 r[4], s; };
      KG kn[NC];
      Q8fRaw raw;                                    // (the q rows in front of the K rows: loads return in order)
      if (tid < 256) {
        if constexpr (NR == 4) raw.v[0] = reinterpret_cast<const f4 *>(qrows(0) + (size_t)w * a.qs)[lane];
        else q8f_fetch(tid, qrows, a.qs, raw);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (append && w == 7) append_new();          // (the other waves do not wait for this one's K rows)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int64_t ro = krow(16 * (w + 8 * c) + lr);
        const u32x4 *src = reinterpret_cast<const u32x4 *>(a.L.kd + ro * KRB + 16 * lq);
#pragma unroll
        for (int j = 0; j < 4; ++j) kn[c].r[j] = src[4 * j];
        kn[c].s = *reinterpret_cast<const u32x4 *>(a.L.ks + ro * kScaleRowBytes);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (tid < 256) {
        if constexpr (NR == 4) {
          reinterpret_cast<f4 *>(&s_q4[w % kGqa][0])[lane] = raw.v[0];
          __builtin_amdgcn_wave_barrier();           // (wave h reads what it wrote: row h)
          q8lim_build(&s_q4[0][0], kHd, reinterpret_cast<int8_t *>(s_p), s_lt, &s_wide, tid, 256);
        } else {
          q8f_digits(tid, raw, reinterpret_cast<uint4 *>(s_p), s_lo2, s_ex, &s_flags, &s_wide);
        }
      }
      lds_barrier();
      const bool wide = s_wide != 0u;
      const unsigned flags = (unsigned)__builtin_amdgcn_readfirstlane((int)s_flags);
      const int lim = lq < nqv ? (int)a.pos0 + q0 + lq : -1;         // (NR 16) the last key of query lq
      h8 da[2][8];
      Q8Lim ql;
      // Lanes 32.. of a chunk's first 8 bytes and lanes ..31 of its second change places: then word pair 0
      // holds block 2 j, word pair 1 block 2 j + 1, lane group lq dims 8 pq .. + 7 of either.
      const int pq = ((lq & 1) << 1) | (lq >> 1);
      if constexpr (NR == 4) {
        q8lim_load(reinterpret_cast<const int8_t *>(s_p), s_lt, ql, pq);
      } else {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int b = 0; b < 8; ++b) da[j][b] = __builtin_bit_cast(h8, reinterpret_cast<const uint4 *>(s_p)[(j * 8 + b) * 64 + 16 * pq + lr]);
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int kg = w + 8 * c, key = 16 * kg + lr;
        if (16 * kg >= kend) break;                  // (wave-uniform)
        long kb8[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const auto x = __builtin_amdgcn_permlane32_swap(kn[c].r[j][0], kn[c].r[j][2], false, false);
          const auto y = __builtin_amdgcn_permlane32_swap(kn[c].r[j][1], kn[c].r[j][3], false, false);
          kb8[2 * j] = (long)((unsigned long)x[0] | ((unsigned long)y[0] << 32));
          kb8[2 * j + 1] = (long)((unsigned long)x[1] | ((unsigned long)y[1] << 32));
        }
        u32x4 ksc = kn[c].s;
        if (append && kg == (kend - 1) >> 4 && key == kend - 1) {
#pragma unroll
          for (int b = 0; b < 8; ++b) kb8[b] = reinterpret_cast<const long *>(&s_row[0][0])[4 * b + pq];
          ksc = *reinterpret_cast<const u32x4 *>(&s_row[0][16]);
        }
        if constexpr (NR == 4) {
          float v;
          if (!wide) {
            v = q8_score16r(kb8, make_uint4(ksc[0], ksc[1], ksc[2], ksc[3]), ql.a, ql.t);
          } else {
            float r[4];
            const int64_t ro = krow(key);
            const bool nw = append && key == kend - 1;
            q8_score_key_slow(nw ? reinterpret_cast<const uint32_t *>(&s_row[0][0]) : reinterpret_cast<const uint32_t *>(a.L.kd + ro * KRB),
                              nw ? reinterpret_cast<const uint32_t *>(&s_row[0][16])
                                 : reinterpret_cast<const uint32_t *>(a.L.ks + ro * kScaleRowBytes), qrows(0), a.qs, r);
            v = lq == 0 ? r[0] : lq == 1 ? r[1] : lq == 2 ? r[2] : r[3];
          }
          v *= a.scale;
          if (key < kend) {
            s_sc[lq][key] = v;
            mx[0] = fmaxf(mx[0], v);
          }
        } else {
          float r[4];
          if (!wide) {
            const f4 z = {0.f, 0.f, 0.f, 0.f};
            const uint32_t sw[4] = {ksc[0], ksc[1], ksc[2], ksc[3]};
            float x[8][4];
            h8 kb[8];
#pragma unroll
            for (int b = 0; b < 8; ++b) {
              const uint32_t w0 = (uint32_t)kb8[b] ^ 0x80808080u, w1 = (uint32_t)((unsigned long)kb8[b] >> 32) ^ 0x80808080u;
              kb[b] = __builtin_bit_cast(h8, make_uint4(as_u(bytes_h2<0x04010400u>(w0)), as_u(bytes_h2<0x04030402u>(w0)),
                                                        as_u(bytes_h2<0x04010400u>(w1)), as_u(bytes_h2<0x04030402u>(w1))));
              const f4 s0 = mfma16(da[0][b], kb[b], z), s1 = mfma16(da[1][b], kb[b], z);
              x[b][0] = __builtin_fmaf(s0[1], 0x1p-8f, s0[0]);
              x[b][1] = __builtin_fmaf(s0[3], 0x1p-8f, s0[2]);
              x[b][2] = __builtin_fmaf(s1[1], 0x1p-8f, s1[0]);
              x[b][3] = __builtin_fmaf(s1[3], 0x1p-8f, s1[2]);
            }
            if (flags != 0u) {
#pragma unroll
              for (int b = 0; b < 8; ++b) {
                if (flags & (1u << b)) {             // a third digit
                  const f4 s0 = mfma16(da[0][b], kb[b], z), s1 = mfma16(da[1][b], kb[b], z);
                  const f4 s2 = mfma16(__builtin_bit_cast(h8, s_lo2[b * 64 + 16 * pq + lr]), kb[b], z);
                  x[b][0] = (float)__builtin_fma((double)s2[0], 0x1p-14, __builtin_fma((double)s0[1], 0x1p-8, (double)s0[0]));
                  x[b][1] = (float)__builtin_fma((double)s2[1], 0x1p-14, __builtin_fma((double)s0[3], 0x1p-8, (double)s0[2]));
                  x[b][2] = (float)__builtin_fma((double)s2[2], 0x1p-14, __builtin_fma((double)s1[1], 0x1p-8, (double)s1[0]));
                  x[b][3] = (float)__builtin_fma((double)s2[3], 0x1p-14, __builtin_fma((double)s1[3], 0x1p-8, (double)s1[2]));
                }
              }
            }
#pragma unroll
            for (int b = 0; b < 8; ++b) {
              const float sf = f16_half(sw[b >> 1], b & 1);
#pragma unroll
              for (int k = 0; k < 4; ++k) r[k] = b == 0 ? __builtin_fmaf(sf, x[0][k], 0.0f) : __fadd_rn(r[k], __fmul_rn(sf, x[b][k]));
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) r[k] *= s_ex[4 * lq + k];
          } else {
            const int64_t ro = krow(key);
            q8_score_key_slow(reinterpret_cast<const uint32_t *>(a.L.kd + ro * KRB),
                              reinterpret_cast<const uint32_t *>(a.L.ks + ro * kScaleRowBytes), qrows(lq), a.qs, r);
          }
          if (key < kend) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const float v = key <= lim ? r[k] * a.scale : -INFINITY;
              s_sc[(4 * lq + k) % NR][key] = v;      // (% NR: the other instantiation's index in range)
              mx[k] = fmaxf(mx[k], v);
            }
          }
        }
      }
    };
    if (kend <= 128) scores(std::integral_constant<int, 1>{});
    else if (kend <= 256) scores(std::integral_constant<int, 2>{});
    else if (kend <= 384) scores(std::integral_constant<int, 3>{});
    else scores(std::integral_constant<int, 4>{});
    if constexpr (NR == 4) {
      const float m = row16_max(mx[0]);
      if (lr == 0) s_red[w][lq] = m;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float m = row16_max(mx[k]);
        if (lr == 0) s_red[w][(4 * lq + k) % NR] = m;
      }
    }
  } else {
    // fp16 K: the reference's serial chain, lane = key 64 w + lane, 32 dimensions (64 B) of its row at a
    // time, two chunks in flight. NR 4: v_mfma_f32_4x4x1 (lane = key, accumulator = head; A = q16 of head
    // lane % 4); NR 16: v_mfma_f32_16x16x1_4b (bkv_mfma16.h).
    const int key = 64 * w + lane;
    const bool mine = 64 * w < kend;               // (wave-uniform)
    const uint4 *src = reinterpret_cast<const uint4 *>(a.L.kd + krow(key) * KRB);
    uint4 kc[2][4];
    auto load = [&](int c, uint4 (&k)[4]) {
#pragma unroll
      for (int i = 0; i < 4; ++i) k[i] = src[4 * c + i];
    };
    constexpr int QL = ((kHd / 4) * NR + kShNT - 1) / kShNT;      // q loads per thread, in front of the K rows
    float4 *s_q = reinterpret_cast<float4 *>(s_p);   // [d4][row]: q16 of dims 4 d4 .. + 3
    float4 qx[QL];
#pragma unroll
    for (int j = 0; j < QL; ++j) {
      const int i = min(tid + j * kShNT, (kHd / 4) * NR - 1), r = i % NR, d4 = i / NR;
      qx[j] = *reinterpret_cast<const float4 *>(qrows(r >> 2) + (size_t)(r & 3) * a.qs + 4 * d4);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (append && w == 7) append_new();
    load(0, kc[0]);                                // (also waves without keys: see above)
    load(1, kc[1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < QL; ++j) {
      const int i = tid + j * kShNT;
      if (i < (kHd / 4) * NR) s_q[i] = make_float4(round_f16(qx[j].x), round_f16(qx[j].y), round_f16(qx[j].z), round_f16(qx[j].w));
    }
    lds_barrier();
    if (mine) {
      f4 d4a = {0.f, 0.f, 0.f, 0.f};
      fv16 d16 = {};
#pragma unroll
      for (int c = 0; c < kHd / 32; ++c) {
        uint4 (&k)[4] = kc[c & 1];
        if (append && key == kend - 1) {
#pragma unroll
          for (int i = 0; i < 4; ++i) k[i] = s_row[0][4 * c + i];
        }
#pragma unroll
        for (int i4 = 0; i4 < 8; ++i4) {
          const float4 q4 = s_q[(8 * c + i4) * NR + (NR == 4 ? (lane & 3) : lr)];
          const float qa[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int i = 4 * i4 + e;
            const float kv = f16_to_f32(half_of(k[i >> 3], i & 7));
            if constexpr (NR == 4) d4a = __builtin_amdgcn_mfma_f32_4x4x1f32(qa[e], kv, d4a, 0, 0, 0);
            else d16 = mfma_k1(qa[e], kv, d16);
          }
        }
        if (c + 2 < kHd / 32) load(c + 2, k);
      }
      if constexpr (NR == 4) {
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const float v = d4a[h] * a.scale;
          if (key < kend) {
            s_sc[h][key] = v;
            mx[h] = v;
          }
        }
      } else {
        const int lim = lq < nqv ? (int)a.pos0 + q0 + lq : -1;
#pragma unroll
        for (int bq = 0; bq < 4; ++bq) {
          const int j = 64 * w + 16 * bq + lr;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const float v = j <= lim ? d16[4 * bq + k] * a.scale : -INFINITY;
            if (j < kend) s_sc[(4 * lq + k) % NR][j] = v;
            mx[k] = fmaxf(mx[k], v);
          }
        }
      }
    }
    if constexpr (NR == 4) {
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const float m = wave_max(mx[h]);
        if (lane == 0) s_red[w][h] = m;
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float m = row16_max(mx[k]);
        if (lr == 0) s_red[w][(4 * lq + k) % NR] = m;
      }
    }
  }

  // ---------------------------------------------------------------- V on its way, e, the serial sums
  const uint32_t vbase = __builtin_amdgcn_readfirstlane(lds_addr(s_v));
  // tile t's rows into buffer t % NB, as prefill_pv64_kernel: 1 KiB blocks of 4 keys x 256 bytes
  auto dma_tile = [&](int t) {
#pragma unroll
    for (int u = 0; u < ND; ++u) {
      const int i = 2 * w + (u & 1);
      const int sw = VF ? (i & 3) : 2 * ((i >> 1) & 3);
      const uint8_t *src = a.L.vd + krow(64 * t + 4 * i + (lane & 3)) * VRB + 256 * (u >> 1) + 16 * ((lane >> 2) ^ sw);
      asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src),
                   "s"(__builtin_amdgcn_readfirstlane(vbase + (uint32_t)VB * (uint32_t)(t % NB) + 1024u * (i + 16 * (u >> 1))))
                   : "memory", "m0");
    }
  };
  const int sw = (w + 7) & 7;                      // the tile whose scale rows this wave takes (wave 0: the eighth)
  if constexpr (VF) {
    if (sw < nt) {
      const uint8_t *src = a.L.vs + krow(64 * sw + lane) * kScaleRowBytes;
      asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src),
                   "s"(__builtin_amdgcn_readfirstlane(lds_addr(s_vs) + 1024u * (uint32_t)sw)) : "memory", "m0");
    }
  }
  for (int t = 0; t < min(nt, NB); ++t) dma_tile(t);
  lds_barrier();                                   // the scores and the waves' maxima
  constexpr int TPR = kShNT / NR;                  // threads per row
  const int er = tid / TPR, ek = tid % TPR, nk64 = 64 * nt;
  float *erow = s_sc[er];
  {
    float m = s_red[0][er];
#pragma unroll
    for (int i = 1; i < 8; ++i) m = fmaxf(m, s_red[i][er]);
    if ((er >> 2) >= nqv) m = 0.0f;                // a row of no query: e = 0
    constexpr int B = 4;                           // exps together: their chains interleave
    for (int k0 = ek; k0 < nk64; k0 += B * TPR) {
      float x[B], e[B];
      bool slow[B], any = false;
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int k = k0 + i * TPR;
        x[i] = k < kend ? erow[k] - m : 0.0f;
      }
#pragma unroll
      for (int i = 0; i < B; ++i) {
        e[i] = exp_t_fast(x[i], s_t2, slow[i]);
        any = any || slow[i];
      }
      if (any) {
#pragma unroll
        for (int i = 0; i < B; ++i)
          if (slow[i]) e[i] = exp_t_slow(x[i]);
      }
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int k = k0 + i * TPR;
        if (k < nk64) erow[k] = k < kend ? e[i] : 0.0f;
        if (NR == 4 && a.e && k < kend) a.e[(size_t)(g * kGqa + er) * a.ld + k] = e[i];
      }
    }
  }
  lds_barrier();
  if (w == 0) {
    // lane r: row r, four keys per read, the next 16 reads in flight (entries past kend are + 0)
    const float4 *row = reinterpret_cast<const float4 *>(s_sc[lane % NR]);
    float sum = 0.0f;
    float4 cur[8], nxt[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) cur[i] = row[i];
    for (int k = 0; k < nk64 / 4; k += 16) {
#pragma unroll
      for (int i = 0; i < 8; ++i) nxt[i] = row[k + 8 + i];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        sum = sum + cur[i].x; sum = sum + cur[i].y; sum = sum + cur[i].z; sum = sum + cur[i].w;
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) cur[i] = row[min(k + 16 + i, nk64 / 4 - 1)];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        sum = sum + nxt[i].x; sum = sum + nxt[i].y; sum = sum + nxt[i].z; sum = sum + nxt[i].w;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (lane < NR) {
      s_sum[lane] = (lane >> 2) < nqv ? sum : 1.0f;
      if (NR == 4) {
        a.sum[g * kGqa + lane] = sum;
        a.status[g * kGqa + lane] = 0u;
      }
    }
  }
  if (VF && (w > 0 || nt == 8)) {
    // Beside the serial sums: the scale rows have landed. (The appended token's, also for the padding after it:
    // those entries were loaded from its slot, which may have held anything, and p = 0 times a NaN scale is NaN.)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (append && sw == (kend - 1) >> 6 && lane >= ((kend - 1) & 63)) s_vs[64 * sw + lane] = s_row[1][16];
    const uint4 s = s_vs[64 * sw + lane];
    if (sw < nt && __any((scale_big(s.x) | scale_big(s.y) | scale_big(s.z) | scale_big(s.w)) != 0u)) s_big = 1u;
  }
  if (NR == 4 && a.gate && w > 0) {
    // the gate's factors beside the serial sums (fp64 exps and divisions: 2 us behind the PV)
    for (int i = tid - 64; i < NR * kHd; i += kShNT - 64)
      s_gate[i % (NR == 4 ? NR * kHd : 4)] = 1.0f / (1.0f + exp_cr(-a.gate[(size_t)(g * kGqa + i / kHd) * a.gs + i % kHd]));
  }
  lds_barrier();
  {
    const float s = s_sum[er], rs = 1.0f / s;
    for (int k = ek; k < nk64; k += TPR)
      *reinterpret_cast<_Float16 *>(s_p + er * kShPS + 2 * k) = (_Float16)div_by_sum(erow[k], s, rs);
  }

  // ---------------------------------------------------------------- PV (as prefill_pv64_kernel, one row tile)
  uint32_t vrd[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    if constexpr (VF) {
      const int j = lr >> 1, bl = 8 * ks + 2 * lq + (j >> 2);
      vrd[ks] = (uint32_t)(1024 * bl + 16 * (j & 3) + 8 * (lane & 1) + 64 * (bl & 3));
    } else {
      const int bl = 8 * ks + 2 * lq;
      vrd[ks] = (uint32_t)(1024 * (bl + 16 * (w >> 2)) + 64 * (((lane >> 1) & 1) ^ (2 * (lq & 3))) + 16 * (lr >> 2) +
                           8 * (lane & 1));
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the first NB tiles have landed
  lds_barrier();                                   // every wave's rows, and p16
  const int lim0 = (int)a.pos0 + q0;               // the first query's last key
  auto rows = [&](int t, int ks) { return *reinterpret_cast<const h8 *>(s_p + lr * kShPS + 2 * (64 * t + 32 * ks + 8 * lq)); };
  // the V operand in pairs of keys (see pv_tile_careful)
  auto ops = [&](int t, int ks, int mt, uint32_t (&x)[4], uint32_t (&s)[4]) {
    const uint32_t vb = vbase + (uint32_t)VB * (uint32_t)(t % NB) + vrd[ks];
    if constexpr (VF) {
      const uint16_t *vs = reinterpret_cast<const uint16_t *>(&s_vs[64 * t + 32 * ks + 8 * lq]) + w;
      const v2i_t bv = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
          (__attribute__((address_space(3))) v2i_t *)(uintptr_t)(vb ^ (uint32_t)(64 * (2 * w + mt))));
      constexpr uint32_t kSel[4] = {0x0C010C00u, 0x0C030C02u, 0x0C050C04u, 0x0C070C06u};
#pragma unroll
      for (int pp = 0; pp < 4; ++pp) {
        const uint32_t bw = __builtin_amdgcn_perm((uint32_t)bv.y, (uint32_t)bv.x, kSel[pp]) ^ 0x64806480u;
        x[pp] = as_u(as_h2(bw) - h2{(_Float16)1152.0f, (_Float16)1152.0f});
        s[pp] = (uint32_t)vs[16 * pp] | ((uint32_t)vs[16 * pp + 8] << 16);
      }
    } else {
      const uint32_t ad = vb ^ (uint32_t)(128 * (2 * (w & 3) + mt));
      const v4s_t r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s_t *)(uintptr_t)ad);
      const v4s_t r1 =
          __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s_t *)(uintptr_t)(ad + 1024u));
      const uint4 v = __builtin_bit_cast(uint4, (v8s_t){r0[0], r0[1], r0[2], r0[3], r1[0], r1[1], r1[2], r1[3]});
      x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    }
  };
  // Chains per value by tile (mod NS) and key half, and the small parts of q8_0 products on their own: the
  // matrix cores round every step of a chain down (see the header). (The loop takes NS tiles a turn: chosen by a
  // branch at the end of a tile instead, a decode of 300 keys takes 13.2 to 14.0 us, not 12.8.)
  constexpr int NS = 3;
  f4 zh[NS][2][2] = {}, zl[2][1] = {};             // [tile mod NS][key half][mt]; [mt]
  auto careful = [&](int t) {
    f4 z[2][1] = {{zh[0][0][0]}, {zh[0][0][1]}};
    uint32_t x[2][2][4], s[2][4];                  // (requested together)
#pragma unroll
    for (int i = 0; i < 4; ++i) ops(t, i >> 1, i & 1, x[i >> 1][i & 1], s[i >> 1]);
    pv_tile_careful<VF, 1, NQ>(
        z, zl, 64 * t, lim0, 64 * t + 63 > lim0,
        [&](int ks, int mt, uint32_t (&xk)[4], uint32_t (&sk)[4]) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            xk[i] = ks ? x[1][mt][i] : x[0][mt][i];
            sk[i] = ks ? s[1][i] : s[0][i];
          }
        },
        [&](int ks, int) { return rows(t, ks); });
    zh[0][0][0] = z[0][0];
    zh[0][0][1] = z[1][0];
  };
  unsigned later = 0;                              // fp16 V: tiles that need pv_tile_careful (of this wave's dims)
  // Tile t's values in its buffer: tile t + NB - 1 goes into tile t - 1's buffer once every wave has read that
  // one; later tiles are waited for in order, the younger ones' loads left in flight.
  auto arrive = [&](int t) {
    if (t > 0 && nt > NB) {
      if (t >= NB) {
        if (t + 1 >= nt) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(ND) : "memory");
      }
      lds_barrier();
      if (t + NB - 1 < nt) dma_tile(t + NB - 1);
    }
    char *vt = s_v[t % NB];
    if (append && t == nt - 1) {                   // the appended row, this wave's dims, over its loaded copy
      const int r = (kend - 1) & 63;
      if constexpr (VF) {
        const int i = r >> 2;
        if (lane < 2)
          *reinterpret_cast<uint4 *>(vt + 1024 * i + 64 * ((2 * w + lane) ^ (i & 3)) + 16 * (r & 3)) = s_row[1][2 * w + lane];
      } else {                                     // (and over the padding's copies: see the scales)
        const int c = 4 * (w & 3) + (lane & 3);
        for (int rr = r + (lane >> 2); rr < 64; rr += 16) {
          const int i = rr >> 2;
          *reinterpret_cast<uint4 *>(vt + 1024 * (i + 16 * (w >> 2)) + 64 * (c ^ (2 * ((i >> 1) & 3))) + 16 * (rr & 3)) =
              s_row[1][4 * w + (lane & 3)];
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  };
  auto tile = [&](int t, f4 (&zp)[2][2]) {
    arrive(t);
    uint32_t x[2][2][4], s[2][4];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) ops(t, ks, mt, x[ks][mt], s[ks]);
    if (!VF && 64 * t + 63 > lim0) {               // some rows do not see some of the tile's keys
      uint32_t nf = 0;
#pragma unroll
      for (int i = 0; i < 16; ++i) nf |= non_finite(x[i >> 3][(i >> 2) & 1][i & 3]);
      if (__any(nf != 0u)) {
        later |= 1u << t;
        return;
      }
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const h8 bp = rows(t, ks);
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const uint32_t (&xk)[4] = x[ks][mt];
        if constexpr (VF) {
          uint32_t hw[4], lw[4];
#pragma unroll
          for (int pp = 0; pp < 4; ++pp) {
            h2 hi, lo;
            split_prod(as_h2(xk[pp]), as_h2(s[ks][pp]), hi, lo);
            hw[pp] = as_u(hi);
            lw[pp] = as_u(lo);
          }
          zp[ks][mt] = mfma16(__builtin_bit_cast(h8, make_uint4(hw[0], hw[1], hw[2], hw[3])), bp, zp[ks][mt]);
          zl[mt][0] = mfma16(__builtin_bit_cast(h8, make_uint4(lw[0], lw[1], lw[2], lw[3])), bp, zl[mt][0]);
        } else {
          zp[ks][mt] = mfma16(__builtin_bit_cast(h8, make_uint4(xk[0], xk[1], xk[2], xk[3])), bp, zp[ks][mt]);
        }
      }
    }
  };
  if (__builtin_expect(VF && s_big != 0u, 0)) {    // a scale past the plain products: a loop of its own
    for (int t = 0; t < nt; ++t) {
      arrive(t);
      careful(t);
    }
  } else {
    for (int t = 0; t < nt; t += NS) {
      tile(t, zh[0]);
      if (t + 1 < nt) tile(t + 1, zh[1]);
      if (NS == 3 && t + 2 < nt) tile(t + 2, zh[NS - 1]);
    }
  }
  if constexpr (!VF)                               // (the last two tiles at most, still in their buffers)
    for (int t = 0; later != 0u; ++t, later >>= 1)
      if (later & 1u) careful(t);
  f4 o[2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt) {
    o[mt] = (zh[0][0][mt] + zh[0][1][mt]) + (zh[1][0][mt] + zh[1][1][mt]);
    if constexpr (NS == 3) zl[mt][0] = (zh[2][0][mt] + zh[2][1][mt]) + zl[mt][0];
    o[mt] = o[mt] + zl[mt][0];
  }
  // lane l holds out^T[dim 32 w + 16 mt + 4 lq + i][row lr] in o[mt][i]
  if (lr < NR && (lr >> 2) < nqv) {
    const size_t row = (size_t)(q0 + (lr >> 2)) * a.nh + g * kGqa + (lr & 3);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const int d = 32 * w + 16 * mt + 4 * lq;
      const float4 v = make_float4(o[mt][0], o[mt][1], o[mt][2], o[mt][3]);
      *reinterpret_cast<float4 *>(a.out + row * kHd + d) = v;
      if (a.gate) {
        float4 f;
        if constexpr (NR == 4) {
          f = *reinterpret_cast<const float4 *>(&s_gate[lr * kHd + d]);
        } else {
          const float4 gt = *reinterpret_cast<const float4 *>(a.gate + row * a.gs + d);
          f = make_float4(1.0f / (1.0f + exp_cr(-gt.x)), 1.0f / (1.0f + exp_cr(-gt.y)), 1.0f / (1.0f + exp_cr(-gt.z)),
                          1.0f / (1.0f + exp_cr(-gt.w)));
        }
        *reinterpret_cast<float4 *>(a.out_gated + row * kHd + d) = make_float4(v.x * f.x, v.y * f.y, v.z * f.z, v.w * f.w);
      }
    }
  }
}

hipError_t launch_short(const ShortArgs &a, int kf, int vf, hipStream_t st) {
  const bool pg = a.L.page != 0;
  BKV_FMT_SWITCH(kf, vf, {
    if (a.n_q == 1) {
      if (pg) hipLaunchKernelGGL((short_kernel<KF_, VF_, 4, true>), dim3(a.nkv), dim3(kShNT), 0, st, a);
      else hipLaunchKernelGGL((short_kernel<KF_, VF_, 4, false>), dim3(a.nkv), dim3(kShNT), 0, st, a);
    } else {
      const dim3 grid(a.nkv * ((a.n_q + 3) / 4));
      if (pg) hipLaunchKernelGGL((short_kernel<KF_, VF_, 16, true>), grid, dim3(kShNT), 0, st, a);
      else hipLaunchKernelGGL((short_kernel<KF_, VF_, 16, false>), grid, dim3(kShNT), 0, st, a);
    }
  });
  return hipGetLastError();
}

}  // namespace bkv
