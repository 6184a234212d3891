// bkv_prefill.hip - chunked prefill attention on the gfx950 matrix cores (bkv_attn_prefill_chunk).
//
// Query i of the chunk (position pos0 + i) attends causally to keys 0 .. pos0 + i, exactly the row
// bkv_attn_decode computes with nfill = pos0 + i + 1 (the reference's prefill is that decode row
// repeated, runtime_vk/attn_vk.h:261-311 per token; bonsai_forward.h:2752-2759). Rows are (query,
// head) pairs; the 4 query heads of one KV head share every K/V tile read.
//
// Work split: a workgroup owns 16 queries x 4 heads = 64 rows of one KV group and one contiguous
// range of 64-key tiles (a "split"); splits exist only to fill the chip when the chunk is short.
// Two passes over the same tiles:
//   stats  S^T = K . Q^T per tile on MFMA, masked causally; online (max, sum exp) per row,
//          written per split;
//   pv     the splits' statistics give the row max M and sum S; scores recomputed bit-identically,
//          p16 = f16(exp(s*scale - M) / S) (the reference rounds the normalised probability to
//          fp16 before PV, attn_vk.h:184-189), then out^T = V^T . P^T on MFMA;
//   merge  (more than one split) the normalised partial outputs are summed in split order, and the
//          gate applied.
//
// Exactness of the matrix-core operands: Q is rounded to fp16 as the reference does; a q8_0 K or V
// element d*b (fp16 scale d, int8 b) has up to 18 significant bits, so it enters the MFMA as the
// exact fp16 pair hi = f16(d*b), lo = d*b - hi (the rounding error of an fp16 product is an fp16
// number, computed by one fp16 fma), and fp16 x fp16 products are exact in the fp32 accumulator.
// What differs from the serial reference is only the order of the fp32 sums (dot products, the
// softmax sum and PV), hence a tolerance rather than bit-exact parity for prefill.

#include <type_traits>

#include "bkv_device.h"
#include "bkv_exp.h"
#include "bkv_internal.h"
#include "bkv_mfma16.h"
#include "bkv_pv8.h"

namespace bkv {

constexpr int kPfNT = 256;      // 4 waves
constexpr int kPfRS = 144;      // LDS row stride in bytes of the P and V^T tiles (64 fp16 + pad)

// exp(x) for x <= 0 (or -inf) in fp32 to about 2 ulp: 2^(x log2 e) on the hardware exp2 with the
// rounding error of the product x*log2(e) carried as a first-order correction
__device__ __forceinline__ float fexp(float x) {
  x = fmaxf(x, -150.0f);
  constexpr float L = 0x1.715476p0f;          // log2(e) rounded to float
  constexpr float Llo = 1.925963033e-8f;      // log2(e) - L
  const float t = x * L;
  const float err = fmaf(x, L, -t) + x * Llo;
  const float y = __builtin_amdgcn_exp2f(t);
  return fmaf(y, err * 0.6931471806f, y);
}

struct PfGeo {
  int g, s, qb, q0, nqv, t0, t1;
  uint32_t kend;
};

// blockIdx -> (KV group, split, query block). Workgroups are dealt to the 8 XCDs round-robin; when
// the grid is a multiple of 8 the index is permuted so that one XCD runs consecutive query blocks
// of one (group, split), which read the same K/V tiles through that XCD's L2.
__device__ __forceinline__ PfGeo pf_geo(const PrefillArgs &a) {
  const int n = gridDim.x, b = blockIdx.x;
  const int i = (n & 7) == 0 ? (b & 7) * (n >> 3) + (b >> 3) : b;
  PfGeo p;
  p.qb = i % a.nqb;
  p.s = (i / a.nqb) % a.nsplit;
  p.g = i / (a.nqb * a.nsplit);
  p.q0 = p.qb * kPfQ;
  p.nqv = min(kPfQ, a.n_q - p.q0);
  p.kend = a.pos0 + (uint32_t)(p.q0 + p.nqv);
  const int nt = (int)((p.kend + kPfTile - 1) / kPfTile);
  p.t0 = (int)((int64_t)p.s * nt / a.nsplit);
  p.t1 = (int)((int64_t)(p.s + 1) * nt / a.nsplit);
  return p;
}

// Q fragments (MFMA B operand of S^T = K.Q^T): row-tile nt, k-step s, lane l holds Q[row 16nt +
// l%16][dims 64(l/16) + 8s .. + 8] in fp16 (rounded to nearest even)
__device__ __forceinline__ void load_q(const PrefillArgs &a, const PfGeo &p, int lane, h8 (&qf)[4][8]) {
  const int lr = lane & 15, lq = lane >> 4;
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    const int r = 16 * nt + lr;
    const int qi = min(p.q0 + (r >> 2), a.n_q - 1);
    const float *qp = a.q + ((size_t)qi * a.nh + (size_t)(p.g * kGqa + (r & 3))) * a.qs + 64 * lq;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const float4 x0 = *reinterpret_cast<const float4 *>(qp + 8 * s);
      const float4 x1 = *reinterpret_cast<const float4 *>(qp + 8 * s + 4);
      h8 h;
      h[0] = (_Float16)x0.x; h[1] = (_Float16)x0.y; h[2] = (_Float16)x0.z; h[3] = (_Float16)x0.w;
      h[4] = (_Float16)x1.x; h[5] = (_Float16)x1.y; h[6] = (_Float16)x1.z; h[7] = (_Float16)x1.w;
      qf[nt][s] = h;
    }
  }
}

// the raw K bytes one lane feeds to the MFMA for a tile: key kb + l%16, dims 64(l/16) .. + 64
template <int KF>
struct KRaw {
  uint4 d[KF ? 4 : 8];
  uint32_t sc;                  // q8_0: the scales of blocks 2(l/16), 2(l/16)+1
};

template <int KF, bool PG>
__device__ __forceinline__ void load_k(const LayerView &L, int nkv, int g, uint32_t key, int lq,
                                       KRaw<KF> &r) {
  const int64_t sl = slot_t<PG>(L, key);
  constexpr int RB = row_bytes(KF ? BKV_Q8_0 : BKV_F16);
  const uint4 *src = reinterpret_cast<const uint4 *>(L.kd + (sl * nkv + g) * RB + (RB / 4) * lq);
#pragma unroll
  for (int c = 0; c < (KF ? 4 : 8); ++c) r.d[c] = src[c];
  if constexpr (KF)
    r.sc = *reinterpret_cast<const uint32_t *>(L.ks + (sl * nkv + g) * kScaleRowBytes + 4 * lq);
}

// S^T tile (16 keys of this wave x 64 rows): acc[nt][i] = dot(K[key 4(l/16)+i], Q[row 16nt + l%16])
template <int KF>
__device__ __forceinline__ void qk_tile(const KRaw<KF> &r, const h8 (&qf)[4][8], f4 (&acc)[4]) {
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) acc[nt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    if constexpr (KF) {
      const uint32_t w0 = r.d[s >> 1][(s & 1) * 2] ^ 0x80808080u;
      const uint32_t w1 = r.d[s >> 1][(s & 1) * 2 + 1] ^ 0x80808080u;
      const uint32_t sw = s < 4 ? (r.sc & 0xFFFFu) * 0x10001u : (r.sc >> 16) * 0x10001u;
      const h2 sc = as_h2(sw);
      h2 hi[4], lo[4];
      split_prod(bytes_h2<0x04010400u>(w0), sc, hi[0], lo[0]);
      split_prod(bytes_h2<0x04030402u>(w0), sc, hi[1], lo[1]);
      split_prod(bytes_h2<0x04010400u>(w1), sc, hi[2], lo[2]);
      split_prod(bytes_h2<0x04030402u>(w1), sc, hi[3], lo[3]);
      const h8 ah = {hi[0][0], hi[0][1], hi[1][0], hi[1][1], hi[2][0], hi[2][1], hi[3][0], hi[3][1]};
      const h8 al = {lo[0][0], lo[0][1], lo[1][0], lo[1][1], lo[2][0], lo[2][1], lo[3][0], lo[3][1]};
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        acc[nt] = mfma16(ah, qf[nt][s], acc[nt]);
        acc[nt] = mfma16(al, qf[nt][s], acc[nt]);
      }
    } else {
      const h8 ak = __builtin_bit_cast(h8, r.d[s]);
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) acc[nt] = mfma16(ak, qf[nt][s], acc[nt]);
    }
  }
}

// causal limit of the lane's rows: the last key row 16nt + l%16 may see (-1: no such query)
__device__ __forceinline__ void row_limits(const PrefillArgs &a, const PfGeo &p, int lr, int (&lim)[4]) {
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    const int r = 16 * nt + lr;
    lim[nt] = (r >> 2) < p.nqv ? (int)(a.pos0 + (uint32_t)(p.q0 + (r >> 2))) : -1;
  }
}

// ------------------------------------------------------------------ pass 1: row statistics
template <int KF, bool PG>
__global__ __launch_bounds__(kPfNT) void prefill_stats_kernel(PrefillArgs a) {
  const PfGeo p = pf_geo(a);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lq = lane >> 4;
  __shared__ float2 s_st[4][4][64];

  h8 qf[4][8];
  load_q(a, p, lane, qf);
  int lim[4];
  row_limits(a, p, lr, lim);
  float m[4], l[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) { m[nt] = -3.0e38f; l[nt] = 0.f; }

  const uint32_t klast = p.kend - 1;
  KRaw<KF> cur, nxt;
  if (p.t0 < p.t1) load_k<KF, PG>(a.L, a.nkv, p.g, min((uint32_t)(p.t0 * kPfTile + 16 * w + lr), klast), lq, cur);
  for (int t = p.t0; t < p.t1; ++t) {
    const int tn = min(t + 1, p.t1 - 1);
    load_k<KF, PG>(a.L, a.nkv, p.g, min((uint32_t)(tn * kPfTile + 16 * w + lr), klast), lq, nxt);
    f4 acc[4];
    qk_tile<KF>(cur, qf, acc);
    const int kb = t * kPfTile + 16 * w + 4 * lq;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      float v[4], mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = kb + i <= lim[nt] ? acc[nt][i] * a.scale : -INFINITY;
        mx = fmaxf(mx, v[i]);
      }
      const float mn = fmaxf(m[nt], mx);
      float sum = l[nt] * fexp(m[nt] - mn);
#pragma unroll
      for (int i = 0; i < 4; ++i) sum += fexp(v[i] - mn);
      m[nt] = mn;
      l[nt] = sum;
    }
    cur = nxt;
  }
  // the four lanes holding one row (l%16 equal), then the four waves
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) s_st[w][lq][16 * nt + lr] = make_float2(m[nt], l[nt]);
  __syncthreads();
  if (tid < 64) {
    float mm = -3.0e38f;
#pragma unroll
    for (int k = 0; k < 16; ++k) mm = fmaxf(mm, s_st[k >> 2][k & 3][tid].x);
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const float2 e = s_st[k >> 2][k & 3][tid];
      ss += e.y * fexp(e.x - mm);
    }
    if ((tid >> 2) < p.nqv) {
      const size_t row = (size_t)(p.q0 + (tid >> 2)) * a.nh + p.g * kGqa + (tid & 3);
      a.stats[(size_t)p.s * a.n_q * a.nh + row] = make_float2(mm, ss);
    }
  }
}

// ------------------------------------------------------------------ pass 2: probabilities and PV
template <int VF>
struct VRaw {
  uint4 a[VF ? 2 : 4], b[VF ? 2 : 4];   // keys 2kp, 2kp+1: dims 64w + 32h .. + 32
  uint32_t sa, sb;                       // q8_0: their scales (fp16 bits in the low half)
};

template <int VF, bool PG>
__device__ __forceinline__ void load_v(const LayerView &L, int nkv, int g, uint32_t ka, uint32_t kb,
                                       int w, int h, VRaw<VF> &r) {
  const int64_t sa = slot_t<PG>(L, ka), sb = slot_t<PG>(L, kb);
  constexpr int RB = row_bytes(VF ? BKV_Q8_0 : BKV_F16);
  constexpr int DB = VF ? 1 : 2;   // bytes per element
  const int off = (64 * w + 32 * h) * DB;
  const uint4 *pa = reinterpret_cast<const uint4 *>(L.vd + (sa * nkv + g) * RB + off);
  const uint4 *pb = reinterpret_cast<const uint4 *>(L.vd + (sb * nkv + g) * RB + off);
#pragma unroll
  for (int c = 0; c < (VF ? 2 : 4); ++c) { r.a[c] = pa[c]; r.b[c] = pb[c]; }
  if constexpr (VF) {
    const int blk = 2 * w + h;
    r.sa = *reinterpret_cast<const uint16_t *>(L.vs + (sa * nkv + g) * kScaleRowBytes + 2 * blk);
    r.sb = *reinterpret_cast<const uint16_t *>(L.vs + (sb * nkv + g) * kScaleRowBytes + 2 * blk);
  }
}

// V^T into the wave's LDS tiles: vt_hi/vt_lo[dim 0..63][key 0..63] (row stride kPfRS), the lane
// writing keys 2kp, 2kp+1 of dims 32h .. + 32
template <int VF>
__device__ __forceinline__ void put_vt(const VRaw<VF> &r, int kp, int h, char *vt_hi, char *vt_lo) {
  char *bh = vt_hi + (32 * h) * kPfRS + 4 * kp;
  if constexpr (VF) {
    char *bl = vt_lo + (32 * h) * kPfRS + 4 * kp;
    const h2 sc = as_h2((r.sa & 0xFFFFu) | (r.sb << 16));
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const uint32_t wa = r.a[c >> 2][c & 3] ^ 0x80808080u, wb = r.b[c >> 2][c & 3] ^ 0x80808080u;
      const uint32_t t0 = __builtin_amdgcn_perm(wb, wa, 0x05010400u);   // a0 b0 a1 b1
      const uint32_t t1 = __builtin_amdgcn_perm(wb, wa, 0x07030602u);   // a2 b2 a3 b3
      const h2 x[4] = {bytes_h2<0x04010400u>(t0), bytes_h2<0x04030402u>(t0),
                       bytes_h2<0x04010400u>(t1), bytes_h2<0x04030402u>(t1)};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        h2 hi, lo;
        split_prod(x[i], sc, hi, lo);
        *reinterpret_cast<uint32_t *>(bh + (4 * c + i) * kPfRS) = as_u(hi);
        *reinterpret_cast<uint32_t *>(bl + (4 * c + i) * kPfRS) = as_u(lo);
      }
    }
  } else {
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const uint32_t wa = r.a[c >> 2][c & 3], wb = r.b[c >> 2][c & 3];
      *reinterpret_cast<uint32_t *>(bh + (2 * c) * kPfRS) = __builtin_amdgcn_perm(wb, wa, 0x05040100u);
      *reinterpret_cast<uint32_t *>(bh + (2 * c + 1) * kPfRS) = __builtin_amdgcn_perm(wb, wa, 0x07060302u);
    }
  }
}

template <int KF, int VF, bool PG>
__global__ __launch_bounds__(kPfNT) void prefill_pv_kernel(PrefillArgs a) {
  const PfGeo p = pf_geo(a);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lq = lane >> 4;
  const int kp = lane & 31, vh = lane >> 5;
  __shared__ __attribute__((aligned(16))) char s_p[2][64 * kPfRS];
  __shared__ __attribute__((aligned(16))) char s_vt[4][VF ? 2 : 1][64 * kPfRS];
  __shared__ float2 s_ms[64];

  // row max and 1/sum from the splits' statistics
  if (tid < 64) {
    float mm = -3.0e38f, ss = 0.f;
    if ((tid >> 2) < p.nqv) {
      const size_t row = (size_t)(p.q0 + (tid >> 2)) * a.nh + p.g * kGqa + (tid & 3);
      const size_t rs = (size_t)a.n_q * a.nh;
      for (int s = 0; s < a.nsplit; ++s) mm = fmaxf(mm, a.stats[s * rs + row].x);
      for (int s = 0; s < a.nsplit; ++s) {
        const float2 e = a.stats[s * rs + row];
        ss += e.y * fexp(e.x - mm);
      }
    }
    s_ms[tid] = make_float2(mm, ss > 0.f ? 1.0f / ss : 0.f);
  }
  h8 qf[4][8];
  load_q(a, p, lane, qf);
  int lim[4];
  row_limits(a, p, lr, lim);
  __syncthreads();
  float M[4], iS[4];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    const float2 e = s_ms[16 * nt + lr];
    M[nt] = e.x;
    iS[nt] = e.y;
  }

  f4 o[4][4];   // [dim tile][row tile]: out^T[dim 64w + 16mt + 4(l/16) + i][row 16nt + l%16]
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) o[mt][nt] = f4{0.f, 0.f, 0.f, 0.f};

  char *vt_hi = s_vt[w][0];
  char *vt_lo = s_vt[w][VF ? 1 : 0];
  const uint32_t klast = p.kend - 1;
  KRaw<KF> kc, kn;
  VRaw<VF> vc, vn;
  auto vkeys = [&](int t, uint32_t &ka, uint32_t &kb) {
    ka = min((uint32_t)(t * kPfTile + 2 * kp), klast);
    kb = min((uint32_t)(t * kPfTile + 2 * kp + 1), klast);
  };
  if (p.t0 < p.t1) {
    load_k<KF, PG>(a.L, a.nkv, p.g, min((uint32_t)(p.t0 * kPfTile + 16 * w + lr), klast), lq, kc);
    uint32_t ka, kb;
    vkeys(p.t0, ka, kb);
    load_v<VF, PG>(a.L, a.nkv, p.g, ka, kb, w, vh, vc);
  }
  int buf = 0;
  for (int t = p.t0; t < p.t1; ++t) {
    const int tn = min(t + 1, p.t1 - 1);
    load_k<KF, PG>(a.L, a.nkv, p.g, min((uint32_t)(tn * kPfTile + 16 * w + lr), klast), lq, kn);
    {
      uint32_t ka, kb;
      vkeys(tn, ka, kb);
      load_v<VF, PG>(a.L, a.nkv, p.g, ka, kb, w, vh, vn);
    }
    f4 acc[4];
    qk_tile<KF>(kc, qf, acc);
    const int kb0 = t * kPfTile + 16 * w + 4 * lq;
    char *pb = s_p[buf];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      h2 pp[2];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = fexp(acc[nt][i] * a.scale - M[nt]) * iS[nt];
        pp[i >> 1][i & 1] = (_Float16)(kb0 + i <= lim[nt] ? e : 0.f);
      }
      *reinterpret_cast<uint2 *>(pb + (16 * nt + lr) * kPfRS + 2 * (16 * w + 4 * lq)) =
          make_uint2(as_u(pp[0]), as_u(pp[1]));
    }
    put_vt<VF>(vc, kp, vh, vt_hi, vt_lo);
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      h8 bp[4];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
        bp[nt] = *reinterpret_cast<const h8 *>(pb + (16 * nt + lr) * kPfRS + 2 * (32 * ks + 8 * lq));
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        const h8 ah = *reinterpret_cast<const h8 *>(vt_hi + (16 * mt + lr) * kPfRS + 2 * (32 * ks + 8 * lq));
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) o[mt][nt] = mfma16(ah, bp[nt], o[mt][nt]);
        if constexpr (VF) {
          const h8 al = *reinterpret_cast<const h8 *>(vt_lo + (16 * mt + lr) * kPfRS + 2 * (32 * ks + 8 * lq));
#pragma unroll
          for (int nt = 0; nt < 4; ++nt) o[mt][nt] = mfma16(al, bp[nt], o[mt][nt]);
        }
      }
    }
    buf ^= 1;
    kc = kn;
    vc = vn;
  }

  // rows' outputs: the final result (one split) or the split's normalised partial
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    const int r = 16 * nt + lr;
    if ((r >> 2) >= p.nqv) continue;
    const size_t row = (size_t)(p.q0 + (r >> 2)) * a.nh + p.g * kGqa + (r & 3);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int d = 64 * w + 16 * mt + 4 * lq;
      const float4 v = make_float4(o[mt][nt][0], o[mt][nt][1], o[mt][nt][2], o[mt][nt][3]);
      if (a.nsplit > 1) {
        *reinterpret_cast<float4 *>(a.part + ((size_t)p.s * a.n_q * a.nh + row) * kHd + d) = v;
      } else {
        *reinterpret_cast<float4 *>(a.out + row * kHd + d) = v;
        if (a.gate) {
          const float4 gt = *reinterpret_cast<const float4 *>(a.gate + row * a.gs + d);
          float4 og;
          og.x = v.x * (1.0f / (1.0f + exp_cr(-gt.x)));
          og.y = v.y * (1.0f / (1.0f + exp_cr(-gt.y)));
          og.z = v.z * (1.0f / (1.0f + exp_cr(-gt.z)));
          og.w = v.w * (1.0f / (1.0f + exp_cr(-gt.w)));
          *reinterpret_cast<float4 *>(a.out_gated + row * kHd + d) = og;
        }
      }
    }
  }
}

// ------------------------------------------------------------------ merge of the splits + gate
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a) {
  const size_t n4 = (size_t)a.n_q * a.nh * (kHd / 4);
  const size_t rs4 = n4;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
    const float4 *pp = reinterpret_cast<const float4 *>(a.part);
    float4 v = pp[i];
    for (int s = 1; s < a.nsplit; ++s) {
      const float4 x = pp[s * rs4 + i];
      v.x += x.x; v.y += x.y; v.z += x.z; v.w += x.w;
    }
    reinterpret_cast<float4 *>(a.out)[i] = v;
    if (a.gate) {
      const float4 gt = *reinterpret_cast<const float4 *>(a.gate + gate_index(4 * i, a.gs));
      float4 og;
      og.x = v.x * (1.0f / (1.0f + exp_cr(-gt.x)));
      og.y = v.y * (1.0f / (1.0f + exp_cr(-gt.y)));
      og.z = v.z * (1.0f / (1.0f + exp_cr(-gt.z)));
      og.w = v.w * (1.0f / (1.0f + exp_cr(-gt.w)));
      reinterpret_cast<float4 *>(a.out_gated)[i] = og;
    }
  }
}

hipError_t launch_prefill(const PrefillArgs &a, int kf, int vf, hipStream_t st) {
  const int grid = a.nkv * a.nqb * a.nsplit;
  const bool pg = a.L.page != 0;
  BKV_FMT_SWITCH(kf, vf, {
    if (pg) {
      hipLaunchKernelGGL((prefill_stats_kernel<KF_, true>), dim3(grid), dim3(kPfNT), 0, st, a);
      hipLaunchKernelGGL((prefill_pv_kernel<KF_, VF_, true>), dim3(grid), dim3(kPfNT), 0, st, a);
    } else {
      hipLaunchKernelGGL((prefill_stats_kernel<KF_, false>), dim3(grid), dim3(kPfNT), 0, st, a);
      hipLaunchKernelGGL((prefill_pv_kernel<KF_, VF_, false>), dim3(grid), dim3(kPfNT), 0, st, a);
    }
  });
  if (a.nsplit > 1) {
    const size_t n4 = (size_t)a.n_q * a.nh * (kHd / 4);
    const int blocks = (int)std::min<size_t>((n4 + 255) / 256, 2048);
    hipLaunchKernelGGL(prefill_merge_kernel, dim3(blocks), dim3(256), 0, st, a);
  }
  return hipGetLastError();
}

// ================================================================== exact prefill
// The default prefill: every (query, head) row reproduces the serial reference bit for bit up to
// the PV contraction. A unit is 4 queries x 4 heads = 16 rows of one KV group; its scores live in a
// scratch region [query][key][4 heads]. Four launches per slice of queries:
//   scores  (q8_0 K: the correctly rounded inner sum of each block, bkv_q8dot.h's contract, then
//           acc = acc + f16(scale)*inner in block order; fp16 K: the reference's serial chain
//           acc = acc + q16*k in ascending d, one exact fma per step on the fp32 matrix cores),
//           times the softmax scale, masked causally; the row maxima. The keys of a unit are split
//           over workgroups so that short chunks fill the chip too.
//   sums    e = exp(v - max) correctly rounded, written back over the scores; one lane per row adds
//           them in key order (the reference's serial fp32 sum, attn_vk.h:175-189).
//   pv      p16 = f16(e / sum) (the correctly rounded fp32 quotient, from e * (1/sum) by two remainder
//           corrections, then round to nearest even), and sum p16 * v on the matrix cores for 128
//           rows (slices of up to 16 queries: 64) and one of pv_split key ranges. Tiles whose V is past
//           the plain products, or not finite where a row does not see the key, take pv_tile_careful.
//   merge   the key ranges' partials added by eights, the eights in fp64, and the gate.
// Only the PV sum runs in another order than the reference (fp32 accumulation of exact products; slices
// of up to 16 queries add their tiles in fp64).

// scratch accesses (plain loads and stores: the scratch round trips are served largely by the
// memory-side cache, which non-temporal accesses bypass)
__device__ __forceinline__ void st_sc4(float *p, float4 v) { *reinterpret_cast<float4 *>(p) = v; }
__device__ __forceinline__ float4 ld_sc4(const float *p) { return *reinterpret_cast<const float4 *>(p); }

// the score kernels' work item: a run of NU units (NU x 4 queries) of one KV group and one of the
// ksplit ranges of its key tiles (TILE keys each). Workgroups are dealt to the 8 XCDs round-robin;
// when the grid is a multiple of 8 the index is permuted so that one XCD runs consecutive query
// blocks of one (group, key range), which read the same K rows through that XCD's L2.
// query block i of n in the order short, long, short, ... (a block's keys grow with its index): an
// XCD's or a round's run of consecutive blocks then has about the same work whatever the start position
__device__ __forceinline__ int px_mix(int i, int n) { return i & 1 ? n - 1 - (i >> 1) : i >> 1; }

struct PxItem {
  int u0, g, s, t0, t1;
  uint32_t kend;                                   // keys 0 .. kend - 1 of the last unit's last query
};
template <int NU, int TILE>
__device__ __forceinline__ PxItem px_item(const PrefillXArgs &a) {
  const int n = gridDim.x, b = blockIdx.x;
  const int wi = (n & 7) == 0 ? (b & 7) * (n >> 3) + (b >> 3) : b;
  const int nub = (a.nqb + NU - 1) / NU;
  PxItem p;
  p.u0 = NU * px_mix(wi % nub, nub);
  p.s = (wi / nub) % a.ksplit;
  p.g = wi / (nub * a.ksplit);
  p.kend = a.pos0 + (uint32_t)min(a.q_base + kPxQ * (p.u0 + NU), a.q_base + a.n_q);
  const int nt = (int)((p.kend + TILE - 1) / TILE);
  p.t0 = (int)((int64_t)p.s * nt / a.ksplit);
  p.t1 = (int)((int64_t)(p.s + 1) * nt / a.ksplit);
  return p;
}

// A workgroup scores UQ units against its range of key tiles (TILE keys each; UQ = 1: 128, else 64).
// The tile's bytes become fp16 B operands in LDS once for all its units (2.5 instructions per 4 bytes:
// at one unit per conversion they were a third of the kernel's VALU work), a tile ahead of the MFMAs:
// lane (key, block) of the 8 waves loads 32 bytes and their scale while the tile before is scored, and
// writes [key group][block][lane] operands (lanes XOR 8 (block % 2), so that the 8-key runs of two
// blocks fall on different banks) and fp32 scales. Wave w scores unit w % UQ against NKG key groups.
template <int UQ, bool PG>
__global__ __launch_bounds__(512, 1) void prefill_score_q8_kernel(PrefillXArgs a) {
  constexpr int TILE = UQ == 1 ? 2 * kPxTile : kPxTile, KGS = TILE / 16, NKG = KGS * UQ / 8, NC = TILE / 64;
  const PxItem p = px_item<UQ, TILE>(a);
  const int tid = threadIdx.x, lane = tid & 63, ql = lane >> 4, n16 = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), u = w % UQ, kg0 = NKG * (w / UQ);
  __shared__ uint4 s_op[2][KGS * 8 * 64];          // first the units' digits (kQ8fUnit each), then the tiles
  __shared__ __attribute__((aligned(16))) float s_sc[2][TILE][8];
  __shared__ uint4 s_lo2[UQ][8 * 64];
  __shared__ float s_ex[UQ][kPxRows];
  __shared__ float s_red[8][kPxRows];
  __shared__ unsigned s_flags[UQ], s_wide;
  static_assert(sizeof(s_op) >= UQ * kQ8fUnit * 16, "the units' digits in the operand buffers");
  uint4 *const op = &s_op[0][0];
  if (tid < UQ) s_flags[tid] = 0u;
  if (tid == 0) s_wide = 0u;
  __syncthreads();
  // (a workgroup's units past the slice's last one repeat that one: the same values stored twice)
  auto unit = [&](int i) { return min(p.u0 + i, a.nqb - 1); };
  const int qlast = a.q_base + a.n_q - 1;
  auto qrows = [&](int q) {                        // the 4 q rows of chunk query q (clamped into the slice)
    return a.q + ((size_t)min(q, qlast) * a.nh + p.g * kGqa) * a.qs;
  };
  for (int i = tid >> 8; i < UQ; i += 2) {
    const int q0 = a.q_base + kPxQ * unit(i);
    Q8fRaw raw;
    q8f_fetch(tid & 255, [&](int q) { return qrows(q0 + q); }, a.qs, raw);
    q8f_digits(tid & 255, raw, op + i * kQ8fUnit, s_lo2[i], s_ex[i], &s_flags[i], &s_wide);
  }
  __syncthreads();
  h8 da[2][8];                                     // the A operands of the wave's unit
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int b = 0; b < 8; ++b) da[j][b] = __builtin_bit_cast(h8, op[u * kQ8fUnit + (j * 8 + b) * 64 + lane]);
  const int uq = kPxQ * unit(u) + ql;              // the lane's query in the slice
  const int lim = uq < a.n_q ? (int)(a.pos0 + (uint32_t)(a.q_base + uq)) : -1;   // the last key it sees
  const unsigned flags = (unsigned)__builtin_amdgcn_readfirstlane((int)s_flags[u]);
  float mx[4], ex[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) { mx[k] = -INFINITY; ex[k] = s_ex[u][4 * ql + k]; }
  constexpr int RB = row_bytes(BKV_Q8_0);
  float *sc = a.sc + (((size_t)(p.g * a.nqb + unit(u)) * kPxQ + ql) * a.ld + n16) * kGqa;
  // the scores of key group kg (keys key0 + 16 kg + lane % 16): lane l holds query l / 16's 4 heads;
  // scaled, masked, into the scratch and the row maxima
  auto emit = [&](uint32_t key0, int kg, const float (&r)[4]) {
    const uint32_t j = key0 + (uint32_t)(16 * kg);
    const bool live = (int)(j + n16) <= lim;
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = live ? r[k] * a.scale : -INFINITY;
      mx[k] = fmaxf(mx[k], v[k]);
    }
    st_sc4(sc + (size_t)j * kGqa, make_float4(v[0], v[1], v[2], v[3]));
  };
  if (s_wide == 0u) {
    __syncthreads();                               // the digits are in registers
    // this lane's (key, block) pairs of a tile: key 64 c + 8 w + lane % 8, block lane / 8
    const int cn = lane & 7, cb = lane >> 3;
    uint4 raw[NC][2];
    uint32_t rsc[NC];
    auto fetch = [&](int t) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const uint32_t key = min((uint32_t)(t * TILE + 64 * c + 8 * w + cn), p.kend - 1);
        const int64_t ro = slot_t<PG>(a.L, key) * a.nkv + p.g;
        const uint4 *src = reinterpret_cast<const uint4 *>(a.L.kd + ro * RB + 32 * cb);
        raw[c][0] = src[0];
        raw[c][1] = src[1];
        rsc[c] = *reinterpret_cast<const uint16_t *>(a.L.ks + ro * kScaleRowBytes + 2 * cb);
      }
    };
    auto convert = [&](int t) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int key = 64 * c + 8 * w + cn;       // of the tile
        uint4 *o = op + (t & 1) * (KGS * 8 * 64) + ((key >> 4) * 8 + cb) * 64;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t w0 = (q & 1 ? raw[c][q >> 1].z : raw[c][q >> 1].x) ^ 0x80808080u;
          const uint32_t w1 = (q & 1 ? raw[c][q >> 1].w : raw[c][q >> 1].y) ^ 0x80808080u;
          o[(16 * q + (key & 15)) ^ (8 * (cb & 1))] =
              make_uint4(as_u(bytes_h2<0x04010400u>(w0)), as_u(bytes_h2<0x04030402u>(w0)),
                         as_u(bytes_h2<0x04010400u>(w1)), as_u(bytes_h2<0x04030402u>(w1)));
        }
        s_sc[t & 1][key][cb] = f16_to_f32(rsc[c]);
      }
    };
    // every block's sums first (independent MFMAs), then the blocks with a third digit again, then the
    // chains
    auto score = [&](auto third, int t, int kg) {
      const f4 z = {0.f, 0.f, 0.f, 0.f};
      const uint4 *kop = op + (t & 1) * (KGS * 8 * 64) + kg * 8 * 64;
      const float4 *sp = reinterpret_cast<const float4 *>(s_sc[t & 1][16 * kg + n16]);
      const float4 sa = sp[0], sb = sp[1];
      float x[8][4];
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        const h8 kb = __builtin_bit_cast(h8, kop[b * 64 + (lane ^ (8 * (b & 1)))]);
        const f4 s0 = mfma16(da[0][b], kb, z), s1 = mfma16(da[1][b], kb, z);
        x[b][0] = __builtin_fmaf(s0[1], 0x1p-8f, s0[0]);
        x[b][1] = __builtin_fmaf(s0[3], 0x1p-8f, s0[2]);
        x[b][2] = __builtin_fmaf(s1[1], 0x1p-8f, s1[0]);
        x[b][3] = __builtin_fmaf(s1[3], 0x1p-8f, s1[2]);
      }
      if constexpr (third.value) {
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          if (flags & (1u << b)) {                 // (wave-uniform)
            const h8 kb = __builtin_bit_cast(h8, kop[b * 64 + (lane ^ (8 * (b & 1)))]);
            const f4 s0 = mfma16(da[0][b], kb, z), s1 = mfma16(da[1][b], kb, z);
            const f4 s2 = mfma16(__builtin_bit_cast(h8, s_lo2[u][b * 64 + lane]), kb, z);
            x[b][0] = (float)__builtin_fma((double)s2[0], 0x1p-14, __builtin_fma((double)s0[1], 0x1p-8, (double)s0[0]));
            x[b][1] = (float)__builtin_fma((double)s2[1], 0x1p-14, __builtin_fma((double)s0[3], 0x1p-8, (double)s0[2]));
            x[b][2] = (float)__builtin_fma((double)s2[2], 0x1p-14, __builtin_fma((double)s1[1], 0x1p-8, (double)s1[0]));
            x[b][3] = (float)__builtin_fma((double)s2[3], 0x1p-14, __builtin_fma((double)s1[3], 0x1p-8, (double)s1[2]));
          }
        }
      }
      const float sf[8] = {sa.x, sa.y, sa.z, sa.w, sb.x, sb.y, sb.z, sb.w};
      float r[4];
#pragma unroll
      for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          r[k] = b == 0 ? __builtin_fmaf(sf[0], x[0][k], 0.0f) : __fadd_rn(r[k], __fmul_rn(sf[b], x[b][k]));
#pragma unroll
      for (int k = 0; k < 4; ++k) r[k] *= ex[k];
      emit((uint32_t)(t * TILE), kg, r);
    };
    // tiles in descending key order (the sums kernel reads them ascending)
    auto sweep = [&](auto third) {
      fetch(p.t1 - 1);
      convert(p.t1 - 1);
      lds_barrier();
      for (int t = p.t1 - 1; t >= p.t0; --t) {
        if (t > p.t0) fetch(t - 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < NKG; ++c) score(third, t, kg0 + c);
        __builtin_amdgcn_sched_barrier(0);
        if (t > p.t0) convert(t - 1);              // (the buffer of tile t + 1, read before the last barrier)
        lds_barrier();
      }
    };
    if (p.t0 < p.t1) {                             // (the same barriers in both)
      if (flags == 0u) sweep(std::false_type{});
      else sweep(std::true_type{});
    }
  } else {
    // the fp64 path: lane = key 16 kg + l%16 against query l/16's 4 heads
    for (int t = p.t1 - 1; t >= p.t0; --t) {
      for (int kg = kg0; kg < kg0 + NKG; ++kg) {
        const uint32_t key = min((uint32_t)(t * TILE + 16 * kg + n16), p.kend - 1);
        const int64_t ro = slot_t<PG>(a.L, key) * a.nkv + p.g;
        float r[4];
        q8_score_key_slow(reinterpret_cast<const uint32_t *>(a.L.kd + ro * RB),
                          reinterpret_cast<const uint32_t *>(a.L.ks + ro * kScaleRowBytes), qrows(a.q_base + uq), a.qs, r);
        emit((uint32_t)(t * TILE), kg, r);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float m = row16_max(mx[k]);
    if (n16 == 0) s_red[w][4 * ql + k] = m;
  }
  __syncthreads();
  if (tid < UQ * kPxRows) {
    const int i = tid / kPxRows, r = tid % kPxRows;
    float m = s_red[i][r];
#pragma unroll
    for (int k = 1; k < 8 / UQ; ++k) m = fmaxf(m, s_red[i + UQ * k][r]);
    a.mx[((size_t)(p.g * a.nqb + unit(i)) * a.ksplit + p.s) * kPxRows + r] = m;
  }
}

// ---------------------------------------------------------------- fp16 K scores on the matrix cores
// v_mfma_f32_16x16x1_4b_f32 computes, for 4 independent blocks b, D_b[i][j] += A_b[i] * B_b[j] with
// one rounding per element: A_b[i] comes from lane 16b + i, B_b[j] from lane 16b + j, and lane l
// holds D_b[4(l/16) + k][l%16] in accumulator register 4b + k. With K = 1 each step is exactly one
// fp32 fma per element (the product of two fp16 values is exact in fp32), so a chain of steps in
// ascending dimension is the reference's serial score, bit for bit. (q8_0 K: bkv_q8dot.h.)
// A workgroup scores NU units against its range of 256-key tiles: one chain of 256 steps per (row,
// key), acc = acc + q16*k in ascending dimension. Block b of the instruction is key group b (keys 16b ..
// + 15 of the wave's 64), so one MFMA advances 64 keys x 16 rows; the wave's NU units are independent
// chains on the same keys (each key's row, streamed 32 dimensions = 64 B at a time, one chunk ahead, goes
// through the L1 once for all of them: with one unit and two key sets instead, the 64 lines a load
// touches took as long as the MFMAs). s_qh[u][d4][i] = q16 of row i, dims 4 d4 .. + 3 (the lanes of one
// row read the same float4).
template <int NU, bool PG>
__global__ __launch_bounds__(256, 2) void prefill_score_f16_kernel(PrefillXArgs a) {
  const PxItem p = px_item<NU, kPxTile16>(a);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), ql = lane >> 4;
  __shared__ float4 s_qh[NU][(kHd / 4) * kPxRows];
  __shared__ float s_red[4][NU][kPxRows];
  // (a workgroup's units past the slice's last one repeat that one: the same values stored twice)
  auto unit = [&](int i) { return min(p.u0 + i, a.nqb - 1); };
  const int qlast = a.q_base + a.n_q - 1;
#pragma unroll
  for (int u = 0; u < NU; ++u)
    for (int i = tid; i < (kHd / 4) * kPxRows; i += 256) {
      const int r = i & 15, d4 = i >> 4;
      const int qi = min(a.q_base + kPxQ * unit(u) + (r >> 2), qlast);
      const float4 x = *reinterpret_cast<const float4 *>(a.q + ((size_t)qi * a.nh + p.g * kGqa + (r & 3)) * a.qs + 4 * d4);
      s_qh[u][i] = make_float4(round_f16(x.x), round_f16(x.y), round_f16(x.z), round_f16(x.w));
    }
  __syncthreads();
  float *sc[NU], mx[NU][4];
  int lim[NU];                                     // the last key the lane's query sees
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int uq = kPxQ * unit(u) + ql;
    lim[u] = uq < a.n_q ? (int)(a.pos0 + (uint32_t)(a.q_base + uq)) : -1;
    sc[u] = a.sc + ((size_t)(p.g * a.nqb + unit(u)) * kPxQ + ql) * a.ld * kGqa;
#pragma unroll
    for (int k = 0; k < 4; ++k) mx[u][k] = -INFINITY;
  }
  constexpr int RB = row_bytes(BKV_F16);
  struct KChunk { uint4 d[4]; };               // [16 B]: dims 32c .. + 31 of the lane's key
  auto load_chunk = [&](int T, int c, KChunk &k) {
    const uint32_t key = min((uint32_t)(T * kPxTile16 + 64 * w + lane), p.kend - 1);
    const uint4 *src = reinterpret_cast<const uint4 *>(a.L.kd + (slot_t<PG>(a.L, key) * a.nkv + p.g) * RB + 64 * c);
#pragma unroll
    for (int q = 0; q < 4; ++q) k.d[q] = src[q];
  };
  auto chunk = [&](const KChunk &k, int c, fv16 (&d)[NU]) {
#pragma unroll
    for (int i4 = 0; i4 < 8; ++i4) {
      float qa[NU][4];
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const float4 q4 = s_qh[u][(8 * c + i4) * kPxRows + (lane & 15)];
        qa[u][0] = q4.x; qa[u][1] = q4.y; qa[u][2] = q4.z; qa[u][3] = q4.w;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * i4 + e;      // dimension within the chunk: 16-bit half i of the 64 B
        const uint32_t wv = word_of(k.d[i >> 3], (i >> 1) & 3);
        const float kv = f16_to_f32((i & 1) ? (wv >> 16) : (wv & 0xFFFFu));
#pragma unroll
        for (int u = 0; u < NU; ++u) d[u] = mfma_k1(qa[u][e], kv, d[u]);
      }
    }
  };
  KChunk ka, kb;
  // tiles in descending key order (the sums kernel reads them ascending); a wave without a key in the last
  // one leaves it out (nothing reads past the last 64 keys)
  int T = p.t1 - 1;
  if (T >= p.t0 && (uint32_t)(T * kPxTile16 + 64 * w) >= p.kend) --T;
  if (T >= p.t0) load_chunk(T, 0, ka);
  for (; T >= p.t0; --T) {
    fv16 d[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) d[u] = fv16{};
#pragma unroll
    for (int c = 0; c < kHd / 32; c += 2) {
      load_chunk(T, c + 1, kb);
      __builtin_amdgcn_sched_barrier(0);
      chunk(ka, c, d);
      __builtin_amdgcn_sched_barrier(0);
      if (c + 2 < kHd / 32) load_chunk(T, c + 2, ka);
      else load_chunk(max(T - 1, p.t0), 0, ka);
      __builtin_amdgcn_sched_barrier(0);
      chunk(kb, c + 1, d);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) {
#pragma unroll
      for (int bq = 0; bq < 4; ++bq) {
        const uint32_t j = (uint32_t)(T * kPxTile16 + 64 * w + 16 * bq + (lane & 15));
        const bool live = (int)j <= lim[u];
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          v[k] = live ? d[u][4 * bq + k] * a.scale : -INFINITY;
          mx[u][k] = v[k] > mx[u][k] ? v[k] : mx[u][k];
        }
        st_sc4(sc[u] + (size_t)j * kGqa, make_float4(v[0], v[1], v[2], v[3]));
      }
    }
  }
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float m = row16_max(mx[u][k]);
      if ((lane & 15) == 0) s_red[w][u][4 * ql + k] = m;
    }
  __syncthreads();
  if (tid < NU * kPxRows) {
    const int i = tid / kPxRows, r = tid % kPxRows;
    a.mx[((size_t)(p.g * a.nqb + unit(i)) * a.ksplit + p.s) * kPxRows + r] =
        fmaxf(fmaxf(s_red[0][i][r], s_red[1][i][r]), fmaxf(s_red[2][i][r], s_red[3][i][r]));
  }
}

// ---------------------------------------------------------------- exp and the serial sum
// One unit per workgroup of NW waves. Waves 0..NW-2 form e for 64 (NW - 1) keys per step (one key per
// thread, its 16 rows), store them over the scores and into an LDS tile [row][key]; the last wave adds
// the previous step's e values of each row in key order (lane r: row r), four per LDS read and the next
// reads in flight, so the serial chains run beside the exps. The chain bounds short chunks.
template <int NW>
__global__ __launch_bounds__(64 * NW) void prefill_sum_kernel(PrefillXArgs a) {
  constexpr int NT = 64 * NW, kEK = 64 * (NW - 1);    // keys per step
  constexpr int ES = kEK + 4;                         // floats per row of the tile (rows 4 banks apart)
  const int n = gridDim.x, b = blockIdx.x;
  const int wp = (n & 7) == 0 ? (b & 7) * (n >> 3) + (b >> 3) : b;
  const int qb = px_mix(wp % a.nqb, a.nqb);
  const int wi = wp / a.nqb * a.nqb + qb;             // the unit
  const int q0 = a.q_base + qb * kPxQ;                // first query (chunk index)
  const int nqv = min(kPxQ, a.q_base + a.n_q - q0);
  const uint32_t kend = a.pos0 + (uint32_t)(q0 + nqv);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  float *sc = a.sc + (size_t)wi * a.ld * kPxRows;
  __shared__ float s_m[kPxRows];
  __shared__ double s_t2[32];                         // the exp table
  __shared__ __attribute__((aligned(16))) float et[2][kPxRows * ES];
  if (tid < 32) s_t2[tid] = kExp2Tab[tid];
  // the row maxima over the key ranges: 16 lanes of rows per NT / 16 ranges, through the exp tile
  {
    const float *mx = a.mx + (size_t)wi * a.ksplit * kPxRows + (tid & 15);
    float m = -INFINITY;
    for (int s = tid >> 4; s < a.ksplit; s += NT / 16) m = fmaxf(m, mx[s * kPxRows]);
    et[0][tid] = m;
    __syncthreads();
    if (tid < kPxRows) {
      for (int i = 1; i < NT / 16; ++i) m = fmaxf(m, et[0][16 * i + tid]);
      s_m[tid] = (tid >> 2) < nqv ? m : 0.f;
    }
    __syncthreads();
  }
  const int nstep = (int)((kend + kEK - 1) / kEK + 1) & ~1;   // even: the exp waves run steps in pairs
  const uint32_t kscr = (kend + kPxTile - 1) / kPxTile * kPxTile;   // scored keys
  if (w < NW - 1) {
    float mrow[kPxRows];
#pragma unroll
    for (int r = 0; r < kPxRows; ++r) mrow[r] = s_m[r];
    auto fetch = [&](int t, float4 (&v)[kPxRows / 4]) {
      const uint32_t j = min((uint32_t)(t * kEK + tid), kscr - 1);
      const float *src = sc + (size_t)j * kGqa;
#pragma unroll
      for (int q = 0; q < kPxQ; ++q) v[q] = ld_sc4(src + (size_t)q * a.ld * kGqa);
    };
    auto step = [&](int t, const float4 (&vc)[kPxRows / 4]) {
      const uint32_t j = (uint32_t)(t * kEK + tid);
      float *eb = et[t & 1] + tid;
      const bool in = j < kscr;                    // keys past the scores: e = 0 (none are live)
      // all 16 exps first, then the stores: independent exps interleave (their table reads in
      // flight together) instead of each waiting out an LDS round trip behind the stores before it
      float ev[kPxRows], xv[kPxRows];
      bool slow[kPxRows], any = false;
#pragma unroll
      for (int r4 = 0; r4 < kPxRows / 4; ++r4) {
        xv[4 * r4] = vc[r4].x - mrow[4 * r4];
        xv[4 * r4 + 1] = vc[r4].y - mrow[4 * r4 + 1];
        xv[4 * r4 + 2] = vc[r4].z - mrow[4 * r4 + 2];
        xv[4 * r4 + 3] = vc[r4].w - mrow[4 * r4 + 3];
      }
#pragma unroll
      for (int r = 0; r < kPxRows; ++r) {
        ev[r] = exp_t_fast(xv[r], s_t2, slow[r]);
        any = any || slow[r];
      }
      if (any) {
#pragma unroll
        for (int r = 0; r < kPxRows; ++r)
          if (slow[r]) ev[r] = exp_t_slow(xv[r]);
      }
#pragma unroll
      for (int r = 0; r < kPxRows; ++r) eb[r * ES] = in ? ev[r] : 0.f;
      lds_barrier();
      if (in) {
        float *dst = sc + (size_t)j * kGqa;
#pragma unroll
        for (int q = 0; q < kPxQ; ++q)
          st_sc4(dst + (size_t)q * a.ld * kGqa, make_float4(ev[4 * q], ev[4 * q + 1], ev[4 * q + 2], ev[4 * q + 3]));
      }
    };
    // two register sets: each step's scores are requested two steps ahead
    float4 va[kPxRows / 4], vb[kPxRows / 4];
    fetch(0, va);
    __builtin_amdgcn_sched_barrier(0);
    fetch(min(1, nstep - 1), vb);
    for (int t = 0; t < nstep; t += 2) {
      step(t, va);
      __builtin_amdgcn_sched_barrier(0);
      fetch(min(t + 2, nstep - 1), va);
      __builtin_amdgcn_sched_barrier(0);
      step(t + 1, vb);
      __builtin_amdgcn_sched_barrier(0);
      fetch(min(t + 3, nstep - 1), vb);
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
  } else {
    const int r = lane & 15;
    float sum = 0.f;
    lds_barrier();
    for (int t = 0; t < nstep; ++t) {
      const float4 *row = reinterpret_cast<const float4 *>(et[t & 1] + r * ES);
      constexpr int B = 8;                            // reads in flight (32 keys)
      float4 cur[B], nxt[B];
#pragma unroll
      for (int i = 0; i < B; ++i) cur[i] = row[i];
#pragma unroll
      for (int k = 0; k < kEK / 4; k += B) {
        if (k + B < kEK / 4)
#pragma unroll
          for (int i = 0; i < B; ++i) nxt[i] = row[k + B + i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < B; ++i) {
          sum = sum + cur[i].x;
          sum = sum + cur[i].y;
          sum = sum + cur[i].z;
          sum = sum + cur[i].w;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < B; ++i) cur[i] = nxt[i];
      }
      lds_barrier();
    }
    if (lane < kPxRows) a.sums[(size_t)wi * kPxRows + r] = (r >> 2) < nqv ? sum : 1.0f;
  }
}

// out_gated = v * 1/(1 + exp(-gate)) for dims d .. + 3 of the chunk's row
__device__ __forceinline__ void px_gate(const PrefillXArgs &a, size_t row, int d, const float4 &v) {
  const float4 gt = *reinterpret_cast<const float4 *>(a.gate + row * a.gs + d);
  float4 og;
  og.x = v.x * (1.0f / (1.0f + exp_cr(-gt.x)));
  og.y = v.y * (1.0f / (1.0f + exp_cr(-gt.y)));
  og.z = v.z * (1.0f / (1.0f + exp_cr(-gt.z)));
  og.w = v.w * (1.0f / (1.0f + exp_cr(-gt.w)));
  *reinterpret_cast<float4 *>(a.out_gated + row * kHd + d) = og;
}

// ---------------------------------------------------------------- PV
// kPvQ queries (128 rows: query i, head h at row 4 i + h) of one KV group over one of pv_split ranges
// of their key tiles: p16 = f16(e / sum) from the sums kernel's e and sums (the reference's P16,
// attn_vk.h:190-200), out^T = V^T . P^T on v_mfma_f32_16x16x32_f16, wave w of 8 owning dims
// 32 w .. + 31 (one q8_0 block). Each 64-key tile of V goes into LDS by direct-to-LDS loads, 1 KiB
// blocks of 4 keys x 256 bytes (q8_0: whole rows; fp16: the rows' first, then their second halves) in
// the blocked layout of bkv_pv8.h; a lane then reads its A operand (8 keys of one dim) with transposed
// LDS reads. q8_0: one ds_read_b64_tr_b8, and the exact fp16 split of d*b (hi = f16(d*b), lo = d*b -
// hi) forms two operands shared by the 128 rows. fp16: two ds_read_b64_tr_b16. The ranges' partials are
// added in a fixed order by prefill_pv_merge_kernel.
//
// Q = kPvQ / 2, for slices of so few queries: 64 rows, each tile's sums from zero and the tiles added in fp64,
// the small parts of q8_0 products on their own (the fp64 sums of 128 rows would not fit the registers). The
// matrix cores round every step of an fp32 chain down: given p16, one chain per range is 1.6e-7 (6 queries onto
// 3000 keys) to 3.3e-7 (14 onto 64000) from 64 bits, this 9.0e-8 and 1.3e-7, decode rows 1.0e-7 and 1.3e-7. Half
// the rows also take less: 6 onto 3000 11.6 us of 12.2.
template <int VF, bool PG, int Q>
__global__ __launch_bounds__(512, 1) void prefill_pv64_kernel(PrefillXArgs a) {
  constexpr int R = kGqa * Q;                      // rows, Q / kPxQ units' worth
  constexpr int NTR = R / 16;                      // MFMA row tiles
  constexpr int RPW = R / 8;                       // rows per wave of the P tile
  static_assert(kPxRows % RPW == 0, "a wave's rows are a unit or part of one");
  constexpr int WPU = kPxRows / RPW;               // waves per unit
  constexpr bool F64 = Q < kPvQ;
  const int n = gridDim.x, b = blockIdx.x;
  const int nqp = (a.n_q + Q - 1) / Q;
  const int wb = (n & 7) == 0 ? (b & 7) * (n >> 3) + (b >> 3) : b;
  const int qb = px_mix(wb % nqp, nqp), sp = (wb / nqp) % a.pv_split, g = wb / (a.pv_split * nqp);
  const int q0 = a.q_base + Q * qb;                // chunk index of the first query
  const int nqv = min(Q, a.q_base + a.n_q - q0);
  const uint32_t kend = a.pos0 + (uint32_t)(q0 + nqv);
  const int ntl = (int)((kend + kPfTile - 1) / kPfTile);
  const int t0 = (int)((int64_t)sp * ntl / a.pv_split), t1 = (int)((int64_t)(sp + 1) * ntl / a.pv_split);
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  __shared__ __attribute__((aligned(16))) float s_pbuf[2 * R * kPfRS / 4];   // P tiles [row][64 keys] fp16
  char *s_p = reinterpret_cast<char *>(s_pbuf);
  // this thread's probabilities: key pk of a tile, RPW rows of unit xr (whose scratch holds their e
  // up to its own last key kx); the wave's sums in scalar registers
  const int pk = lane;
  const int xr = Q / kPxQ * qb + w / WPU;
  const int xq = min(xr, a.nqb - 1);
  const bool pv = kPxQ * xr < a.n_q;
  const uint32_t kx = a.pos0 + (uint32_t)min(a.q_base + kPxQ * xr + kPxQ, a.q_base + a.n_q);
  const size_t xw = (size_t)g * a.nqb + xq;
  const float *esrc = a.sc + (xw * kPxQ + RPW / kGqa * (w % WPU)) * a.ld * kGqa;
  float ssum[RPW], srcp[RPW];
  f4 o[2][NTR];                                    // (F64: one tile's)
  f4 ol[2][F64 ? NTR : 1];                         // F64, q8_0: the products' small parts, all tiles
  auto zero = [&]() {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int nt = 0; nt < NTR; ++nt) o[mt][nt] = f4{0.f, 0.f, 0.f, 0.f};
  };
  zero();
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < (F64 ? NTR : 1); ++nt) ol[mt][nt] = f4{0.f, 0.f, 0.f, 0.f};
  double tot[2][F64 ? NTR : 1][4] = {};
  auto add = [&]() {
    if constexpr (F64) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int nt = 0; nt < NTR; ++nt)
#pragma unroll
          for (int i = 0; i < 4; ++i) tot[mt][nt][i] += (double)o[mt][nt][i];
    }
  };
  // V tiles: three LDS buffers (tile t in buffer t % 3), each of 16 (fp16: 32) blocks of 1 KiB: 16-byte
  // chunk c of row r of block i at 64 (c ^ swizzle(i)) + 16 r, so that the rows one transposed read
  // takes spread over the banks
  constexpr int VB = VF ? 16384 : 32768;           // bytes per tile
  __shared__ __attribute__((aligned(1024))) char s_v[3][VB];
  const uint32_t vbase = __builtin_amdgcn_readfirstlane(lds_addr(s_v));
  // the lane's read address in a tile buffer for key half ks (q8_0: dim tile mt by XOR 64 (2 w + mt);
  // fp16: dim tile mt by XOR 128 (2 (w % 4) + mt), the second 4 of its 8 keys one block on)
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
  // (the loaded values are kept raw until the tile uses them: any arithmetic on them here would
  // make the wave wait for the loads at once)
  struct PvIn {
    float4 en[RPW / 4];                             // e of key pk, the thread's rows (valid if live)
    bool live;
    uint32_t vs;                                    // the block scale of key 32 (l%16 / 8) + 8 lq + l%8
  };
  // (past t1, ahead of the loop's end: tile t1 - 1 again)
  auto load_tile = [&](int tt, PvIn &in) {
    const int t = min(tt, t1 - 1);
    const uint32_t j = (uint32_t)(t * kPfTile + pk);
    const float *src = esrc + (size_t)min(j, kx - 1) * kGqa;
#pragma unroll
    for (int i = 0; i < RPW / 4; ++i) in.en[i] = ld_sc4(src + (size_t)i * a.ld * kGqa);
    in.live = pv && j < kx;
    if constexpr (VF) {
      // one scale load per lane: lane l%16 of each 16-lane row loads key (l%16 / 8, l%8)'s, and the row
      // shares them by DPP broadcasts in the tile
      const uint32_t skey = min((uint32_t)(t * kPfTile + 32 * (lr >> 3) + 8 * lq + (lr & 7)), kend - 1);
      in.vs = *reinterpret_cast<const uint16_t *>(a.L.vs + (slot_t<PG>(a.L, skey) * a.nkv + g) * kScaleRowBytes + 2 * w);
    }
  };
  // the V rows of tile tt (clamped as above) into buffer tt % 3: wave w loads the blocks i of keys
  // 4 i .. + 3 for i = 2 w, 2 w + 1 (lane: key 4 i + lane % 4, chunk (lane / 4) ^ swizzle at 16 lane)
  constexpr int ND = VF ? 2 : 4;                    // loads per wave
  auto dma_tile = [&](int tt) {
    const int t = min(tt, t1 - 1);
#pragma unroll
    for (int u = 0; u < ND; ++u) {
      const int i = 2 * w + (u & 1);                // block of keys; u / 2: half of an fp16 row
      const uint32_t key = min((uint32_t)(t * kPfTile + 4 * i + (lane & 3)), kend - 1);
      const int sw = VF ? (i & 3) : 2 * ((i >> 1) & 3);
      const uint8_t *src = a.L.vd + (slot_t<PG>(a.L, key) * a.nkv + g) * row_bytes(VF ? BKV_Q8_0 : BKV_F16) +
                           256 * (u >> 1) + 16 * ((lane >> 2) ^ sw);
      asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src),
                   "s"(__builtin_amdgcn_readfirstlane(vbase + (uint32_t)VB * (uint32_t)(tt % 3) + 1024u * (i + 16 * (u >> 1))))
                   : "memory", "m0");
    }
  };
  // tile t's p16 into the P buffer pb, its block scales into vsk
  auto probs = [&](const PvIn &in, char *pb, uint32_t (&vsk)[16]) {
    float ev[RPW];
#pragma unroll
    for (int i = 0; i < RPW / 4; ++i) {
      ev[4 * i] = in.en[i].x; ev[4 * i + 1] = in.en[i].y; ev[4 * i + 2] = in.en[i].z; ev[4 * i + 3] = in.en[i].w;
    }
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const _Float16 h = (_Float16)div_by_sum(in.live ? ev[i] : 0.0f, ssum[i], srcp[i]);
      *reinterpret_cast<_Float16 *>(pb + (RPW * w + i) * kPfRS + 2 * pk) = h;
    }
    // the block scales of the lane's 16 keys: key (ks, c) from lane 8 ks + c of its row
    if constexpr (VF) {
#define BKV_BC(i) vsk[i] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)in.vs, 0x150 + (i), 0xF, 0xF, false)
      BKV_BC(0); BKV_BC(1); BKV_BC(2); BKV_BC(3); BKV_BC(4); BKV_BC(5); BKV_BC(6); BKV_BC(7);
      BKV_BC(8); BKV_BC(9); BKV_BC(10); BKV_BC(11); BKV_BC(12); BKV_BC(13); BKV_BC(14); BKV_BC(15);
#undef BKV_BC
    }
  };
  // tile t's V values of key half ks and dim tile mt as LDS holds them, and from them the operand in pairs of
  // keys (see pv_tile_careful): pair p holds keys 2p, 2p+1 of the lane's 8
  auto vread = [&](int t, int ks, int mt) {
    const uint32_t vb = vbase + (uint32_t)VB * (uint32_t)(t % 3) + (ks ? vrd[1] : vrd[0]);
    if constexpr (VF) {
      const v2i_t bv = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
          (__attribute__((address_space(3))) v2i_t *)(uintptr_t)(vb ^ (uint32_t)(64 * (2 * w + mt))));
      return make_uint4((uint32_t)bv.x, (uint32_t)bv.y, 0u, 0u);
    } else {
      // keys 8 lq .. + 3 of the half from one block, + 4 .. + 7 from the next (the same swizzle)
      const uint32_t ad = vb ^ (uint32_t)(128 * (2 * (w & 3) + mt));
      const v4s_t r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s_t *)(uintptr_t)ad);
      const v4s_t r1 =
          __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s_t *)(uintptr_t)(ad + 1024u));
      return __builtin_bit_cast(uint4, (v8s_t){r0[0], r0[1], r0[2], r0[3], r1[0], r1[1], r1[2], r1[3]});
    }
  };
  auto operand = [&](const uint4 &v, int ks, const uint32_t (&vsk)[16], uint32_t (&x)[4], uint32_t (&s)[4]) {
    if constexpr (VF) {
      constexpr uint32_t kSel[4] = {0x0C010C00u, 0x0C030C02u, 0x0C050C04u, 0x0C070C06u};
#pragma unroll
      for (int pp = 0; pp < 4; ++pp) {
        const uint32_t bw = __builtin_amdgcn_perm(v.y, v.x, kSel[pp]) ^ 0x64806480u;
        x[pp] = as_u(as_h2(bw) - h2{(_Float16)1152.0f, (_Float16)1152.0f});
        s[pp] = ks ? vsk[8 + 2 * pp] | (vsk[9 + 2 * pp] << 16) : vsk[2 * pp] | (vsk[1 + 2 * pp] << 16);
      }
    } else {
      x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    }
  };
  const int lim0 = (int)(a.pos0 + (uint32_t)q0);   // the first query's last key
  __shared__ __attribute__((aligned(8))) uint8_t s_careful[2][8];   // [t % 2][wave]: tile t needs pv_tile_careful
  // true: the tile was left out, as it needs pv_tile_careful
  auto tile = [&](int t, const PvIn &in) {
    char *pb = s_p + (t & 1) * (R * kPfRS);
    uint32_t vsk[16];
    probs(in, pb, vsk);
    if constexpr (VF) {
      const bool big = __any(scale_big(in.vs) != 0u);
      if (lane == 0) s_careful[t & 1][w] = big;
    }
    // this wave's V rows of tile t have landed when at most the loads issued after them are in
    // flight: tile t + 1's register loads (NL) and rows (ND), tile t + 2's register loads (NL)
    constexpr int NL = RPW / 4 + (VF ? 1 : 0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NL + ND) : "memory");
    const bool masked = kPfTile * t + kPfTile - 1 > lim0;   // some rows do not see some of the tile's keys
    if (!VF && masked) {                            // the values this wave loaded
      uint32_t nf = 0;
#pragma unroll
      for (int u = 0; u < ND; ++u) {
        const uint4 v = *reinterpret_cast<const uint4 *>(s_v[t % 3] + 1024 * (2 * w + (u & 1) + 16 * (u >> 1)) + 16 * lane);
        nf |= non_finite(v.x) | non_finite(v.y) | non_finite(v.z) | non_finite(v.w);
      }
      const bool bad = __any(nf != 0u);
      if (lane == 0) s_careful[t & 1][w] = bad;
    }
    lds_barrier();                                  // the P tile and every wave's V rows of tile t
    dma_tile(t + 2);                                // (its buffer's last readers, tile t - 1, are done)
    unsigned long careful = 0;
    if (VF || masked) careful = *reinterpret_cast<const unsigned long *>(s_careful[t & 1]);
    uint4 v[2][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i >> 1][i & 1] = vread(t, i >> 1, i & 1);
    if (__builtin_expect(__builtin_amdgcn_readfirstlane((int)(careful | (careful >> 32))) != 0, 0)) return true;
    // the A operands (registers only)
    h8 ah[2][2], al[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        uint32_t x[4], s[4];
        operand(v[ks][mt], ks, vsk, x, s);
        if constexpr (VF) {
          uint32_t hw[4], lw[4];
#pragma unroll
          for (int pp = 0; pp < 4; ++pp) {
            h2 hi, lo;
            split_prod(as_h2(x[pp]), as_h2(s[pp]), hi, lo);
            hw[pp] = as_u(hi);
            lw[pp] = as_u(lo);
          }
          ah[ks][mt] = __builtin_bit_cast(h8, make_uint4(hw[0], hw[1], hw[2], hw[3]));
          al[ks][mt] = __builtin_bit_cast(h8, make_uint4(lw[0], lw[1], lw[2], lw[3]));
        } else {
          ah[ks][mt] = __builtin_bit_cast(h8, make_uint4(x[0], x[1], x[2], x[3]));
        }
      }
    }
    auto rows = [&](int ks, int nt) { return *reinterpret_cast<const h8 *>(pb + (16 * nt + lr) * kPfRS + 2 * (32 * ks + 8 * lq)); };
#pragma unroll
    for (int nt = 0; nt < NTR; ++nt) {
      const h8 b0 = rows(0, nt), b1 = rows(1, nt);
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        f4 &l = F64 ? ol[mt][F64 ? nt : 0] : o[mt][nt];
        if constexpr (VF) l = mfma16(al[0][mt], b0, l);
        o[mt][nt] = mfma16(ah[0][mt], b0, F64 ? f4{0.f, 0.f, 0.f, 0.f} : o[mt][nt]);
        if constexpr (VF) l = mfma16(al[1][mt], b1, l);
        o[mt][nt] = mfma16(ah[1][mt], b1, o[mt][nt]);
      }
    }
    add();
    return false;
  };
  // three register sets and V buffers, each tile's operands requested two tiles ahead (groups of three
  // without joining branches, so that the compiler's wait counting keeps the two younger tiles' loads in
  // flight); the V rows of tile t + 2 go out once every wave has passed tile t's barrier
  if (t0 < t1) {
    PvIn in[3];
    int tc = t1;                                    // the first tile that needs pv_tile_careful
    load_tile(t0, in[0]);
    dma_tile(t0);
    load_tile(t0 + 1, in[1]);
    dma_tile(t0 + 1);
    // (the sums behind the first tiles' loads, which do not need them)
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      ssum[i] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(
                                              __builtin_bit_cast(int, a.sums[xw * kPxRows + RPW * (w % WPU) + i])));
      srcp[i] = 1.0f / ssum[i];
    }
    for (int t = t0; t < t1; t += 3) {
#pragma unroll
      for (int u = 0; u < 3; ++u) {
        if (u > 0 && t + u >= t1) break;
        load_tile(t + u + 2, in[(u + 2) % 3]);
        __builtin_amdgcn_sched_barrier(0);
        if (tile(t + u, in[u])) {                   // (the same in every wave)
          tc = t + u;
          t = t1;
          break;
        }
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last rows landed before the LDS is used again or released
    // from that tile on one after the other
#pragma unroll 1
    for (int t = tc; t < t1; ++t) {
      lds_barrier();                                // the buffers' last readers are done
      uint32_t vsk[16];
      load_tile(t, in[0]);
      dma_tile(t);
      probs(in[0], s_p, vsk);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      lds_barrier();
      auto &l = [&]() -> f4 (&)[2][NTR] {
        if constexpr (F64) return ol;
        else return o;
      }();
      if constexpr (F64) zero();
      pv_tile_careful<VF, NTR, kPxQ>(
          o, l, kPfTile * t, lim0, kPfTile * t + kPfTile - 1 > lim0,
          [&](int ks, int mt, uint32_t (&x)[4], uint32_t (&s)[4]) { operand(vread(t, ks, mt), ks, vsk, x, s); },
          [&](int ks, int nt) { return *reinterpret_cast<const h8 *>(s_p + (16 * nt + lr) * kPfRS + 2 * (32 * ks + 8 * lq)); });
      add();
    }
  }
  // lane l holds out^T[dim 32 w + 16 mt + 4(l/16) + r][row 16 nt + l%16] in o[mt][nt][r]: the range's
  // partial, or (one range) the output
  const bool whole = a.pv_split == 1;
  float *part = whole ? a.out + (size_t)a.q_base * a.nh * kHd : a.part + (size_t)sp * a.n_q * a.nh * kHd;
#pragma unroll
  for (int nt = 0; nt < NTR; ++nt) {
    const int r = 16 * nt + lr;
    if ((r >> 2) >= nqv) continue;
    const size_t row = (size_t)(q0 - a.q_base + (r >> 2)) * a.nh + g * kGqa + (r & 3);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const int d = 32 * w + 16 * mt + 4 * lq;
      float4 v = make_float4(o[mt][nt][0], o[mt][nt][1], o[mt][nt][2], o[mt][nt][3]);
      if constexpr (F64) {
        double x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = tot[mt][nt][i] + (double)ol[mt][nt][i];
        v = make_float4((float)x[0], (float)x[1], (float)x[2], (float)x[3]);
      }
      *reinterpret_cast<float4 *>(part + row * kHd + d) = v;
      if (whole && a.gate) px_gate(a, (size_t)a.q_base * a.nh + row, d, v);
    }
  }
}

// out = the key ranges' partials (8 requested together and added pairwise, the eights in fp64), and the gate
__global__ __launch_bounds__(256) void prefill_pv_merge_kernel(PrefillXArgs a) {
  const size_t n4 = (size_t)a.n_q * a.nh * (kHd / 4);
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const f4 *pp = reinterpret_cast<const f4 *>(a.part) + i;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  for (int s = 0; s < a.pv_split; s += 8) {
    f4 y[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) y[u] = s + u < a.pv_split ? pp[(size_t)(s + u) * n4] : f4{0.f, 0.f, 0.f, 0.f};
    const f4 t = ((y[0] + y[1]) + (y[2] + y[3])) + ((y[4] + y[5]) + (y[6] + y[7]));
    s0 += (double)t[0]; s1 += (double)t[1]; s2 += (double)t[2]; s3 += (double)t[3];
  }
  const float4 v = make_float4((float)s0, (float)s1, (float)s2, (float)s3);
  const size_t grow = (size_t)a.q_base * a.nh + i / (kHd / 4);   // row of the whole chunk
  const int d = 4 * (int)(i % (kHd / 4));
  *reinterpret_cast<float4 *>(a.out + grow * kHd + d) = v;
  if (a.gate) px_gate(a, grow, d, v);
}

// How many key ranges to split each of `items` work items of `tiles` key tiles into: the count whose
// rounds of `slots` resident workgroups take least, a workgroup costing `fixed` (its prologue and
// epilogue) plus `tile` per tile, and `merge` per range where there are several (ns).
static int px_ranges(int64_t items, int64_t tiles, int64_t slots, int64_t tile, int64_t fixed, int64_t merge, int64_t most) {
  int64_t best = 1, cost = INT64_MAX;
  for (int64_t ks = 1; ks <= std::min<int64_t>({tiles, most, 128}); ++ks) {
    const int64_t c = (items * ks + slots - 1) / slots * ((tiles + ks - 1) / ks * tile + fixed) + (ks > 1 ? ks * merge : 0);
    if (c < cost) {
      cost = c;
      best = ks;
    }
  }
  return (int)best;
}

hipError_t launch_prefill_exact(PrefillXArgs a, int kf, int vf, hipStream_t st) {
  const bool pg = a.L.page != 0;
  const int64_t kmax = (int64_t)a.pos0 + a.q_base + a.n_q;       // keys of the slice's last query
  const int units = a.nkv * a.nqb;
  const int64_t mxmost = (int64_t)kPvSplit * kPxSlice * a.nh * kHd / ((int64_t)units * kPxRows);   // a.mx's space
  // Scores. q8_0: one 8-wave workgroup per CU (its operand tiles fill the LDS); a 64-key tile takes it
  // 2.0 us, the digits and the last stores 7 (512 queries onto 8192 keys: 137 us in one round of 256
  // workgroups, 149 in two, 160 in four; 48 onto 6000: 29 in one, 46 in four). Units a workgroup takes:
  // four where there are that many, so that each tile is converted for all of them.
  if (kf == BKV_Q8_0) {
    const int uq = a.nqb >= 3 ? 4 : a.nqb, tile = uq == 1 ? 2 * kPxTile : kPxTile;
    const int items = a.nkv * ((a.nqb + uq - 1) / uq);
    a.ksplit = px_ranges(items, (kmax + tile - 1) / tile, 256, 2000, 7000, 0, mxmost);
    const dim3 grid(items * a.ksplit);
#define BKV_LAUNCH_SCORE(UQ)                                                                             \
  do {                                                                                                   \
    if (pg) hipLaunchKernelGGL((prefill_score_q8_kernel<UQ, true>), grid, dim3(512), 0, st, a);          \
    else hipLaunchKernelGGL((prefill_score_q8_kernel<UQ, false>), grid, dim3(512), 0, st, a);            \
  } while (0)
    if (uq == 4) BKV_LAUNCH_SCORE(4);
    else if (uq == 2) BKV_LAUNCH_SCORE(2);
    else BKV_LAUNCH_SCORE(1);
#undef BKV_LAUNCH_SCORE
  } else {
    // fp16: 4-wave workgroups of two units (one: a chunk of up to 4 queries), four resident per CU sharing
    // its matrix cores: 24 us for a 256-key tile of each. (300 queries onto 2000 keys: 67 us with every
    // tile a workgroup, 1000 onto none: 75 us, 82-84 with fewer workgroups; 512 onto 8192: 352 us, 392
    // with one unit and two sets of keys per wave.)
    // One unit where the rounds of 256 workgroups then come out shorter (6.8 us a tile, 12.2 with two): 256 onto
    // 500 (768 workgroups of one tile, not 384) 52.3 us for the call, 56.3 with two; 100 onto 1000 47.3, 55.2; 20
    // onto 6000 67.2, 75.3; but 256 onto 700 61.6, 60.6; 1000 onto none 145, 132.
    const int64_t tiles = (kmax + kPxTile16 - 1) / kPxTile16;
    int items = 0;
    auto plan = [&](int nu, int64_t tile) {
      items = a.nkv * ((a.nqb + nu - 1) / nu);
      a.ksplit = px_ranges(items, tiles, 1024, 24000, 2000, 0, mxmost);
      return ((int64_t)items * a.ksplit + 255) / 256 * ((tiles + a.ksplit - 1) / a.ksplit) * tile;
    };
    const bool one = a.nqb == 1 || (units <= 256 && plan(1, 6800) < plan(2, 12200));
    plan(one ? 1 : 2, 0);
    const dim3 grid(items * a.ksplit);
    if (one) {
      if (pg) hipLaunchKernelGGL((prefill_score_f16_kernel<1, true>), grid, dim3(256), 0, st, a);
      else hipLaunchKernelGGL((prefill_score_f16_kernel<1, false>), grid, dim3(256), 0, st, a);
    } else {
      if (pg) hipLaunchKernelGGL((prefill_score_f16_kernel<2, true>), grid, dim3(256), 0, st, a);
      else hipLaunchKernelGGL((prefill_score_f16_kernel<2, false>), grid, dim3(256), 0, st, a);
    }
  }
  // Sums. Up to one unit per CU: 7 exp waves keep up with the chain (48 queries onto 6000 keys: 36 us);
  // more units: 3 exp waves each, several workgroups per CU (512 onto 8192: 127 against 134 us; 300 onto
  // 2000: 30 against 37).
  if (units <= 256) hipLaunchKernelGGL(prefill_sum_kernel<8>, dim3(units), dim3(512), 0, st, a);
  else hipLaunchKernelGGL(prefill_sum_kernel<4>, dim3(units), dim3(256), 0, st, a);
  // PV: one workgroup per CU, 3 us per tile and 8 for the rest (512 onto 8192: 104 us in one round; 48
  // onto 6000: 17 us in one round, 28 in two; 128 onto 500, fp16 V: 10 ranges of one tile 44.4 us for the
  // call, 4 of three 39.8)
  const bool few = a.n_q <= kPvQ / 2;
  const int items = few ? a.nkv : a.nkv * ((a.n_q + kPvQ - 1) / kPvQ);
  // (a range's partials are written and read at about 4 TB/s)
  a.pv_split = px_ranges(items, (kmax + kPfTile - 1) / kPfTile, 256, 3000, 8000, (int64_t)a.n_q * a.nh * kHd * 8 / 4000,
                         kPvSplit * kPxSlice / a.n_q);
  const dim3 pgrid(items * a.pv_split);
#define BKV_LAUNCH_PV(VF, Q)                                                                             \
  do {                                                                                                   \
    if (pg) hipLaunchKernelGGL((prefill_pv64_kernel<VF, true, Q>), pgrid, dim3(512), 0, st, a);          \
    else hipLaunchKernelGGL((prefill_pv64_kernel<VF, false, Q>), pgrid, dim3(512), 0, st, a);            \
  } while (0)
  if (vf == BKV_Q8_0) {
    if (few) BKV_LAUNCH_PV(1, kPvQ / 2);
    else BKV_LAUNCH_PV(1, kPvQ);
  } else {
    if (few) BKV_LAUNCH_PV(0, kPvQ / 2);
    else BKV_LAUNCH_PV(0, kPvQ);
  }
#undef BKV_LAUNCH_PV
  if (a.pv_split == 1) return hipGetLastError();
  const size_t n4 = (size_t)a.n_q * a.nh * (kHd / 4);
  hipLaunchKernelGGL(prefill_pv_merge_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st, a);
  return hipGetLastError();
}

}  // namespace bkv
