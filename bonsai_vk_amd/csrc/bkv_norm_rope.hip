// bkv_norm_rope.hip - the reference's fused append front end (bkv_qk_norm_rope_append): per-head
// RMS norm, weight and rope of the projected Q and K, then K (and the raw V) quantised into the
// cache, Q returned as the fp32 rows the attention rounds to its fp16 operand.
//
// Arithmetic, in the reference's order (runtime_vk/attn_vk.h:102-122, the shader
// runtime_vk/shaders/attn_norm_rope2.comp:138-181):
//   ss = sum over d ascending of (x_d * x_d), each square rounded before it is added;
//   inv = 1 / sqrt(ss / hd + eps)  (correctly rounded division and square root);
//   n_d = (x_d * inv) * w_d;
//   inside the first nrot dims, pair p (p < nrot/2) with p + nrot/2: theta = base^(-2p/nrot) (the
//   exponent formed in fp32), a = pos * theta in fp32, y_p = lo*cos a - hi*sin a,
//   y_{p+nrot/2} = hi*cos a + lo*sin a, every product rounded; dims from nrot on pass through.
// pow, cos and sin are the correctly rounded fp32 values of the exact functions, formed as the
// fp64 library function rounded once to fp32 (the same contract as the softmax's exp). The
// reference's CPU mirror calls the C library's powf/cosf/sinf, which agree with these except where
// a C-library float result is not correctly rounded (one fp32 ulp).

#include "bkv_device.h"
#include "bkv_internal.h"

namespace bkv {

// One workgroup of 8 waves per token and up to kNrGroups KV groups (their Q and K rows in LDS, their V
// rows straight through). One lane per row adds the squares, so the 256-step serial sums of all the
// workgroup's rows run side by side in one wave while two others form the rope's sines (once per token
// and pair) and waves 4.. write the V rows. What bounds it: at one token the chain of latencies (load,
// serial sum, store: 4.0 us; 5.0 with one workgroup per row, whose every row formed its own sines), at 512
// tokens the memory (22 MB: 7.6 us, 15.5 before; 2048 tokens 22 us, 50 before).
constexpr int kNrGroups = 4, kNrRows = 5 * kNrGroups, kNrStride = kHd + 4;

template <int KF, int VF>
__global__ __launch_bounds__(512, 2) void norm_rope_append_kernel(NormRopeArgs a) {
  const int t = blockIdx.x, g0 = kNrGroups * blockIdx.y, ng = min(kNrGroups, a.nkv - g0);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nq = kGqa * ng, nr = nq + ng;        // Q rows, then K rows
  const uint32_t pos = a.pos0 + (uint32_t)t;
  __shared__ __attribute__((aligned(16))) float s_x[kNrRows][kNrStride];
  __shared__ float s_inv[kNrRows], s_cs[kHd / 2], s_sn[kHd / 2];
  const int64_t slot = slot_of(a.L, pos);
  constexpr int RPW = (kNrRows + 7) / 8;         // rows per wave
  // the wave's rows w, w + 8, ..: their values and weights, and the rounded squares into LDS
  float4 xv[RPW], wv[RPW];
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int r = min(w + 8 * j, nr - 1);
    const float *x = r < nq ? a.q_in + ((size_t)t * a.nh + kGqa * g0 + r) * kHd : a.k_in + ((size_t)t * a.nkv + g0 + r - nq) * kHd;
    xv[j] = reinterpret_cast<const float4 *>(x)[lane];
    wv[j] = reinterpret_cast<const float4 *>(r < nq ? a.qn_w : a.kn_w)[lane];
  }
#pragma unroll
  for (int j = 0; j < RPW; ++j)
    if (w + 8 * j < nr)
      reinterpret_cast<float4 *>(s_x[w + 8 * j])[lane] =
          make_float4(xv[j].x * xv[j].x, xv[j].y * xv[j].y, xv[j].z * xv[j].z, xv[j].w * xv[j].w);
  __syncthreads();
  const int half = a.nrot / 2;
  if (w == 0) {
    // lane r adds row r's squares in ascending d, the next 32 read ahead
    const float4 *row = reinterpret_cast<const float4 *>(s_x[min(lane, nr - 1)]);
    float ss = 0.0f;
    float4 cur[8], nxt[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) cur[i] = row[i];
#pragma unroll 1
    for (int k = 0; k < kHd / 4; k += 16) {
#pragma unroll
      for (int i = 0; i < 8; ++i) nxt[i] = row[k + 8 + i];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        ss = ss + cur[i].x; ss = ss + cur[i].y; ss = ss + cur[i].z; ss = ss + cur[i].w;
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) cur[i] = row[min(k + 16 + i, kHd / 4 - 1)];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        ss = ss + nxt[i].x; ss = ss + nxt[i].y; ss = ss + nxt[i].z; ss = ss + nxt[i].w;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (lane < nr) s_inv[lane] = 1.0f / sqrtf(ss / (float)kHd + a.eps);
  } else if (w <= 2) {
    const int p = tid - 64;
    if (p < half) {
      const float ex = -2.0f * (float)p / (float)a.nrot;
      const float th = (float)pow((double)a.freq_base, (double)ex);
      const float ang = (float)pos * th;
      s_cs[p] = (float)cos((double)ang);
      s_sn[p] = (float)sin((double)ang);
    }
  } else if (w >= 4 && w - 4 < ng) {             // V: raw into the cache
    const int h = g0 + w - 4;
    if (lane < 32) {
      uint8_t *dr = const_cast<uint8_t *>(a.L.vd) + (slot * a.nkv + h) * row_bytes(VF);
      uint8_t *sr = VF == BKV_Q8_0 ? const_cast<uint8_t *>(a.L.vs) + (slot * a.nkv + h) * kScaleRowBytes : nullptr;
      append_row<VF, false>(a.v_in + ((size_t)t * a.nkv + h) * kHd, dr, sr, lane);
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int r = w + 8 * j;
    if (r < nr) {
      const float inv = s_inv[r];
      reinterpret_cast<float4 *>(s_x[r])[lane] = make_float4((xv[j].x * inv) * wv[j].x, (xv[j].y * inv) * wv[j].y,
                                                             (xv[j].z * inv) * wv[j].z, (xv[j].w * inv) * wv[j].w);
    }
  }
  __builtin_amdgcn_wave_barrier();               // (from here each wave works on its own rows only)
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int r = w + 8 * j;
    if (r < nr) {
      for (int p = lane; p < half; p += 64) {
        const float cs = s_cs[p], sn = s_sn[p], lo = s_x[r][p], hi = s_x[r][p + half];
        const float l1 = lo * cs, l2 = hi * sn, h1 = hi * cs, h2 = lo * sn;
        s_x[r][p] = l1 - l2;
        s_x[r][p + half] = h1 + h2;
      }
    }
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int j = 0; j < RPW; ++j) {
    const int r = w + 8 * j;
    if (r < nq) {
      reinterpret_cast<float4 *>(a.q_out + ((size_t)t * a.nh + kGqa * g0 + r) * kHd)[lane] =
          reinterpret_cast<const float4 *>(s_x[r])[lane];
    } else if (r < nr && lane < 32) {
      const int h = g0 + r - nq;
      uint8_t *dr = const_cast<uint8_t *>(a.L.kd) + (slot * a.nkv + h) * row_bytes(KF);
      uint8_t *sr = KF == BKV_Q8_0 ? const_cast<uint8_t *>(a.L.ks) + (slot * a.nkv + h) * kScaleRowBytes : nullptr;
      append_row<KF, false>(s_x[r], dr, sr, lane);
    }
  }
}

hipError_t launch_norm_rope_append(const NormRopeArgs &a, int kf, int vf, int n_tok, hipStream_t st) {
  BKV_FMT_SWITCH(kf, vf, hipLaunchKernelGGL((norm_rope_append_kernel<KF_, VF_>),
                                            dim3(n_tok, (a.nkv + kNrGroups - 1) / kNrGroups), dim3(512), 0, st, a));
  return hipGetLastError();
}

}  // namespace bkv
