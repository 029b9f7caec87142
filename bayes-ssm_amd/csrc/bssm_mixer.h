#pragma once
// The Bayes mixer's input transforms and their derivatives (shared by the
// fused kernels of bssm_mixer.hip and bssm_mixer_row.hip).

#include "bssm_rot4.h"

namespace bssm {
namespace r4 {
namespace {

constexpr float kNoiseFloor = 1e-4f;  // softplus(noise) + 1e-4 (train_6layer.py:667-668)
// F.normalize divides by max(|a|, 1e-12): 1 / max(|a|, eps) = min(rsq(|a|^2), 1e12).
constexpr float kInvNormEps = 1e12f;
constexpr float kNormEps2 = 1e-24f;

// The transforms run on the hardware exponential, reciprocal and reciprocal
// square root (v_exp_f32, v_rcp_f32, v_rsq_f32, each within 1 ulp, the
// exponential's argument scaled by log2 e first); the library logf/log1pf
// and the IEEE divide cost 13 to 117 instructions each.
__device__ __forceinline__ float exp_(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }
__device__ __forceinline__ float rcp_(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float sigmoid_(float x) { return rcp_(1.f + exp_(-x)); }

// log(1 + u) for u in [0, 1]: 2 atanh(s) with s = u / (2 + u) <= 1/3, the
// odd series through s^15 (next term below 2e-9 relative).
__device__ __forceinline__ float log1p01(float u) {
  const float s = u * rcp_(2.f + u), z = s * s;
  float p = 1.f / 15.f;
  p = fmaf(p, z, 1.f / 13.f);
  p = fmaf(p, z, 1.f / 11.f);
  p = fmaf(p, z, 1.f / 9.f);
  p = fmaf(p, z, 1.f / 7.f);
  p = fmaf(p, z, 1.f / 5.f);
  p = fmaf(p, z, 1.f / 3.f);
  p = fmaf(p, z, 1.f);
  return 2.f * s * p;
}
// softplus(x) = max(x, 0) + log(1 + e^-|x|) and its derivative sigmoid(x).
// torch's softplus returns x itself above 20, where log(1 + e^-x) < 2.1e-9
// is below half an ulp of x, so the two agree.
__device__ __forceinline__ float softplus_(float x) { return fmaxf(x, 0.f) + log1p01(exp_(-fabsf(x))); }

// The decay exp(-softplus(z)) = 2^-(max(z, 0) log2 e + log2(1 + e^-|z|)),
// with the hardware log2: its absolute error (about 1e-7 in the exponent,
// from rounding 1 + e^-|z|) is one ulp of the decay, so the series of
// log1p01 (which the noise needs for its relative accuracy where softplus is
// tiny) is not needed here.
__device__ __forceinline__ float decay_(float z) {
  const float l = __builtin_amdgcn_logf(1.f + exp_(-fabsf(z)));
  return __builtin_amdgcn_exp2f(-fmaf(fmaxf(z, 0.f), 1.44269504088896341f, l));
}

// silu(x) = x sigmoid(x); silu'(x) = sigmoid(x) (1 + x (1 - sigmoid(x))).
__device__ __forceinline__ float silu_(float x) { return x * sigmoid_(x); }

// normalize(silu(x)) of one head's key or query vector.
__device__ __forceinline__ v4f unit_silu(v4f x) {
  v4f a;
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[i] = silu_(x[i]);
    ss = fmaf(a[i], a[i], ss);
  }
  return a * fminf(__builtin_amdgcn_rsqf(ss), kInvNormEps);
}
// Gradient through normalize(silu(x)): g is dL/d(output).  Above the eps
// clamp, d(a/|a|) = (g - w (w . g)) / |a| with w = a / |a|; below it the map
// is a / eps.
__device__ __forceinline__ v4f unit_silu_grad(v4f x, v4f g) {
  v4f a, ds;
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float sg = sigmoid_(x[i]);
    a[i] = x[i] * sg;
    ds[i] = sg * fmaf(x[i], 1.f - sg, 1.f);
    ss = fmaf(a[i], a[i], ss);
  }
  const float rn = fminf(__builtin_amdgcn_rsqf(ss), kInvNormEps);
  float wg = 0.f;
  if (ss > kNormEps2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) wg = fmaf(a[i] * rn, g[i], wg);
  }
  v4f out;
#pragma unroll
  for (int i = 0; i < 4; ++i) out[i] = fmaf(-a[i] * rn, wg, g[i]) * rn * ds[i];
  return out;
}

__device__ __forceinline__ const float* as_f(const void* p, int64_t bytes) {
  return reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + bytes);
}

// Four bf16 values (a 64-bit piece) to float32, and float32 to a bf16 piece.
__device__ __forceinline__ v4f widen4(v2f piece) {
  const v2u w = __builtin_bit_cast(v2u, piece);
  v4f out;
  out[0] = __builtin_bit_cast(float, w[0] << 16);
  out[1] = __builtin_bit_cast(float, w[0] & 0xffff0000u);
  out[2] = __builtin_bit_cast(float, w[1] << 16);
  out[3] = __builtin_bit_cast(float, w[1] & 0xffff0000u);
  return out;
}
__device__ __forceinline__ v2f narrow4(v4f x) {
  v2u w;
  w[0] = narrow2(x[0], x[1]);
  w[1] = narrow2(x[2], x[3]);
  return __builtin_bit_cast(v2f, w);
}

// Gradient outputs: contiguous [B, T, H * w] rows, bfloat16 or float32.
struct MixGrads {
  Rsrc q, k, v, dl, nz;
  uint32_t rq, rk, rv, rd, rn;  // row bytes of the bf16 layout
  uint32_t ckq, cv, cn;         // byte offset of the wave's first head, bf16 layout
  bool f32;
  __device__ __forceinline__ MixGrads(const MixArgs& a, int64_t bb, int64_t h0) {
    const int64_t T = a.t, H = a.h;
    f32 = a.grad_f32 != 0;
    // Row strides: the caller's, or contiguous rows of 4 / 8 / 2 values per head.
    rq = static_cast<uint32_t>(a.ldgq ? a.ldgq : 4 * H) * 2u;
    rk = static_cast<uint32_t>(a.ldgk ? a.ldgk : 4 * H) * 2u;
    rv = static_cast<uint32_t>(a.ldgv ? a.ldgv : 8 * H) * 2u;
    rd = static_cast<uint32_t>(a.ldgd ? a.ldgd : 4 * H) * 2u;
    rn = static_cast<uint32_t>(a.ldgn ? a.ldgn : 2 * H) * 2u;
    ckq = static_cast<uint32_t>(h0) * 8u;
    cv = static_cast<uint32_t>(h0) * 16u;
    cn = static_cast<uint32_t>(h0) * 4u;
    // Offsets are computed in the bf16 layout; float32 rows are twice as long.
    const int64_t e = f32 ? 2 : 1;
    const uint32_t tq = static_cast<uint32_t>(T * e) * rq, tk = static_cast<uint32_t>(T * e) * rk,
                   tv = static_cast<uint32_t>(T * e) * rv, td = static_cast<uint32_t>(T * e) * rd,
                   tn = static_cast<uint32_t>(T * e) * rn;
    q = make_rsrc(as_f(a.gq, bb * tq), tq);
    k = make_rsrc(as_f(a.gk, bb * tk), tk);
    v = make_rsrc(as_f(a.gv, bb * tv), tv);
    const bool dyn = a.gdl != nullptr;
    dl = make_rsrc(as_f(dyn ? a.gdl : a.gq, dyn ? bb * td : 0), dyn ? td : 0u);
    nz = make_rsrc(as_f(dyn ? a.gnz : a.gq, dyn ? bb * tn : 0), dyn ? tn : 0u);
  }
  // One piece of 8 values (lo = first four, hi = last four) at the bf16
  // byte offset `off`: bf16 as one 16-byte piece, float32 as two.
  __device__ __forceinline__ void put8(Rsrc r, uint32_t off, v4f lo, v4f hi) const {
    if (f32) {
      st128<kNtStore>(r, lo, off < kOob ? 2u * off : kOob, 0);
      st128<kNtStore>(r, hi, off < kOob ? 2u * off + 16u : kOob, 0);
    } else {
      st128<kNtStore>(r, narrow(lo, hi), off, 0);
    }
  }
};

}  // namespace
}  // namespace r4
}  // namespace bssm
