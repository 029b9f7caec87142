// Producer-fused mixer kernels for small batch * heads, gfx950.
//
// The fused kernels of bssm_mixer.hip give a wave 16 heads and need about
// 1024 x 16 sequences to fill the SIMDs; below that the time is one wave's
// instruction stream whatever the batch.  Here a workgroup of three (forward)
// or four (backward) waves holds 4 consecutive heads of one batch row in the
// row layout (bssm_row.h): the covariance and mean waves of the split
// float32 kernels as they are, and a wave of its own for the streams, which
// loads the bfloat16 pieces, applies the input transforms, forms the
// readout's gradient, applies the chain rule and stores.  Its stream is
// shorter than the longest of the others (4 heads to its 64 lanes: in the
// backward one lane a token, head and half), so the transforms hide behind the
// recurrence.
//
// 32 x 511 x 64 heads, gated, through the Python API: forward and backward 275
// us, against 770 us of bssm_mixer.hip's kernels.  T = 511, forward / backward
// of one call in us, here and there: 512 sequences 191 / 306 and 303 / 627; 2048
// 283 / 370 and 374 / 671; 4096 445 / 661 and 498 / 850; 6144 635 / 966 and 639
// / 1071; 8192 806 / 1282 and 782 / 1280 (beyond 2048 a CU's LDS holds one
// backward workgroup of two groups).  Bound by the covariance chain of 35 to 75
// dependent instructions a token.

#include "bssm_mixer.h"
#include "bssm_row.h"

#pragma clang fp contract(off)  // as in bssm_row.h

namespace bssm {
namespace sn {
namespace {

using r4::as_f;
using r4::ld64;
using r4::narrow2;
using r4::narrow4;
using r4::sigmoid_;
using r4::silu_;
using r4::widen4;

__device__ __forceinline__ uint32_t word(float x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ float lo16(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float hi16(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
// Two bf16 values plus their bias, rounded to bf16 once.
__device__ __forceinline__ uint32_t add2(uint32_t x, uint32_t b) {
  return narrow2(lo16(x) + lo16(b), hi16(x) + hi16(b));
}
__device__ __forceinline__ v4f silu4(v4f x) { return v4f{silu_(x[0]), silu_(x[1]), silu_(x[2]), silu_(x[3])}; }

// The 4 heads of a group: batch row, first head, sequence index; none past
// the last group (empty descriptors).
struct Group {
  int64_t bb, h0, n0;
  uint32_t valid;  // 4 or 0
  __device__ __forceinline__ Group(const MixArgs& a, int64_t g) {
    const int64_t hq = a.h / SPW;
    valid = g < a.b * hq ? SPW : 0u;
    if (valid == 0) g = 0;
    bb = g / hq;
    h0 = (g - bb * hq) * SPW;
    n0 = bb * a.h + h0;
  }
};

// Descriptors of the projections of one batch row, which end at token T, and
// their row bytes.
struct Rows {
  Rsrc q, k, v, dl, nz;
  uint32_t rq, rk, rv, rd, rn;
  __device__ __forceinline__ Rows(const MixArgs& a, const Group& g) {
    const int64_t T = a.t;
    auto row = [&](Rsrc& d, uint32_t& bytes, const void* p, int64_t ld) __attribute__((always_inline)) {
      bytes = static_cast<uint32_t>(ld * 2);
      d = make_rsrc(as_f(p, g.bb * T * bytes), g.valid ? static_cast<uint32_t>(T) * bytes : 0u);
    };
    row(q, rq, a.q, a.ldq);
    row(k, rk, a.k, a.ldk);
    row(v, rv, a.v, a.ldv);
    row(dl, rd, a.dl, a.ldd);
    row(nz, rn, a.nz, a.ldn);
  }
};

// G groups of 4 heads per workgroup: waves covariance, mean, streams of each.
template <bool EPI, bool BIAS, int G>
__global__ __launch_bounds__(3 * G * kWave) void mixer_forward_row_kernel(MixArgs a) {
  __shared__ float lds_all[G * STile::SIZE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int role = wave / G, grp = wave % G;
  float* const lds = lds_all + grp * STile::SIZE;
  const int s = lane >> 4, c = lane & 15, i = c >> 2, j = c & 3;
  const int co = 2 * i + (j & 1);
  const bool odd = (j & 1) != 0;
  const float delta = i == j ? 1.f : 0.f;
  const Group g(a, static_cast<int64_t>(blockIdx.x) * G + grp);
  const uint32_t T = static_cast<uint32_t>(a.t);
  const uint32_t nbp = static_cast<uint32_t>(a.nb + 1);
  const uint32_t ntiles = (T + TT - 1) / TT;
  auto in_slot = [&](uint32_t t) __attribute__((always_inline)) {
    return lds + STile::IN + static_cast<int>(t % 3u) * STile::SLOT + s * STile::SEQ;
  };
  auto y_slot = [&](uint32_t t) __attribute__((always_inline)) {
    return lds + STile::Y + static_cast<int>(t & 1u) * STile::YSLOT + s * STile::YSEQ;
  };
  auto bu_slot = [&](uint32_t t) __attribute__((always_inline)) {
    return lds + STile::BU + static_cast<int>(t & 1u) * STile::BSLOT + s * STile::BSEQ;
  };
  auto tile_len = [&](uint32_t t) __attribute__((always_inline)) {
    return static_cast<int>((T - t * TT) < TT ? (T - t * TT) : TT);
  };
  // At step it the streams wave lands tile it + 1 and stores the readouts of
  // tile it - 2, the covariance wave runs tile it, the mean wave tile it - 1.
  if (role == 0) {
    const Rsrc rbc = make_rsrc(a.bc + g.n0 * nbp * 16, g.valid * nbp * 64u);
    const Rsrc rc0 = make_rsrc(a.c0 + g.n0 * 16, g.valid * 64u);
    const Rsrc rcT = make_rsrc(a.cT + g.n0 * 16, g.valid * 64u);
    const uint32_t cvo = static_cast<uint32_t>(s) * 64u + cov_off(i, j);
    const uint32_t cco = static_cast<uint32_t>(s) * nbp * 64u + cov_off(i, j);
    float P = r4::ld32(rc0, cvo, 0);
    r4::vm_wait<0>();
    r4::st32(rbc, P, cco, 0);
    __syncthreads();
    uint32_t next_ckpt = kRot4Chunk, ckpt = 1;
    for (uint32_t it = 0; it <= ntiles; ++it) {
      if (it < ntiles) {
        auto ckpt_at = [&](int tt) __attribute__((always_inline)) {
          if (it * TT + tt == next_ckpt) {
            r4::st32(rbc, P, cco, ckpt * 64u);
            ++ckpt;
            next_ckpt += kRot4Chunk;
          }
        };
        const int len = tile_len(it);
        cov_tile<false>(P, in_slot(it), bu_slot(it), i, j, len, len == TT, delta, a.floor, ckpt_at);
      }
      __syncthreads();
    }
    r4::st32(rcT, P, cvo, 0);
    r4::st32(rbc, P, cco, static_cast<uint32_t>(a.nb) * 64u);
  } else if (role == 1) {
    const Rsrc rbm = make_rsrc(a.bm + g.n0 * nbp * 32, g.valid * nbp * 128u);
    const Rsrc rm0 = make_rsrc(a.m0 + g.n0 * 32, g.valid * 128u);
    const Rsrc rmT = make_rsrc(a.mT + g.n0 * 32, g.valid * 128u);
    const uint32_t mo = static_cast<uint32_t>(s) * 128u + mean_off(i, j);
    const uint32_t cmo = static_cast<uint32_t>(s) * nbp * 128u + mean_off(i, j);
    const v2f m = own_order(ld64(rm0, mo, 0), odd);
    float M0 = m[0], M1 = m[1];
    r4::vm_wait<0>();
    auto own = [&]() __attribute__((always_inline)) {
      v2f x;
      x[0] = M0;
      x[1] = M1;
      return own_order(x, odd);
    };
    r4::st64(rbm, own(), cmo, 0);
    __syncthreads();
    uint32_t next_ckpt = kRot4Chunk, ckpt = 1;
    for (uint32_t it = 0; it <= ntiles; ++it) {
      if (it >= 1) {
        const uint32_t tl = it - 1;
        auto ckpt_at = [&](int tt) __attribute__((always_inline)) {
          if (tl * TT + tt == next_ckpt) {
            r4::st64(rbm, own(), cmo, ckpt * 128u);
            ++ckpt;
            next_ckpt += kRot4Chunk;
          }
        };
        const int len = tile_len(tl);
        mean_tile<false>(M0, M1, in_slot(tl), bu_slot(tl), y_slot(tl), j, co, len, len == TT, ckpt_at);
      }
      __syncthreads();
    }
    r4::st64(rmT, own(), mo, 0);
    r4::st64(rbm, own(), cmo, static_cast<uint32_t>(a.nb) * 128u);
  } else {
    // Lane (s, c): token c of the tile, head s.  Rows past T read zeros and
    // drop their stores (the descriptors' ranges).
    const Rows rows(a, g);
    const uint32_t head = static_cast<uint32_t>(g.h0) + s;
    const uint32_t H = static_cast<uint32_t>(a.h), ro = H * 16u, yrow = H * 32u;
    const uint32_t rg = static_cast<uint32_t>(a.ldg * 2);
    const Rsrc rgate = make_rsrc(EPI ? as_f(a.gate, g.bb * a.t * rg) : a.m0, EPI && g.valid ? T * rg : 0u);
    const Rsrc ryb = make_rsrc(EPI ? as_f(a.yb, g.bb * a.t * ro) : a.m0, EPI && g.valid ? T * ro : 0u);
    const bool precise = a.precise != 0;
    const uint32_t orow = EPI ? (precise ? yrow : ro) : yrow;
    const Rsrc rout = make_rsrc(as_f(EPI ? a.out : a.y, g.bb * a.t * orow), g.valid ? T * orow : 0u);
    uint32_t bd0 = 0, bd1 = 0, bn = 0;
    if constexpr (BIAS) {
      if (g.valid) {
        const uint32_t* ab = static_cast<const uint32_t*>(a.abias);
        bd0 = ab[2 * head];
        bd1 = ab[2 * head + 1];
        bn = ab[2 * H + head];
      }
    }
    v2f xq, xk, xd;
    v4f xv, xg;
    float xn;
    auto load = [&](uint32_t t) __attribute__((always_inline)) {
      const uint32_t tok = t * TT + c;
      xq = ld64(rows.q, tok * rows.rq + head * 8u, 0);
      xk = ld64(rows.k, tok * rows.rk + head * 8u, 0);
      xd = ld64(rows.dl, tok * rows.rd + head * 8u, 0);
      xv = r4::ld128<r4::kNtLoad>(rows.v, tok * rows.rv + head * 16u);
      xn = r4::ld32(rows.nz, tok * rows.rn + head * 4u, 0);
    };
    auto load_gate = [&](uint32_t t) __attribute__((always_inline)) {
      if constexpr (EPI) xg = r4::ld128<r4::kNtLoad>(rgate, (t * TT + c) * rg + head * 16u);
    };
    auto put = [&](uint32_t t) __attribute__((always_inline)) {
      float* b = in_slot(t);
      *reinterpret_cast<v4f*>(b + STile::K + 4 * c) = r4::unit_silu(widen4(xk));
      *reinterpret_cast<v4f*>(b + STile::Q + 4 * c) = r4::unit_silu(widen4(xq));
      uint32_t d0 = word(xd[0]), d1 = word(xd[1]), n = word(xn);
      if constexpr (BIAS) {
        d0 = add2(d0, bd0);
        d1 = add2(d1, bd1);
        n = add2(n, bn);
      }
      *reinterpret_cast<v4f*>(b + STile::D + 4 * c) =
          v4f{r4::decay_(lo16(d0)), r4::decay_(hi16(d0)), r4::decay_(lo16(d1)), r4::decay_(hi16(d1))};
      const v4f v0 = r4::widen_lo(xv), v1 = r4::widen_hi(xv);
      *reinterpret_cast<v4f*>(b + STile::V + 8 * c) = silu4(v0);
      *reinterpret_cast<v4f*>(b + STile::V + 8 * c + 4) = silu4(v1);
      b[STile::P + c] = r4::softplus_(lo16(n)) + r4::kNoiseFloor;
      b[STile::R + c] = r4::softplus_(hi16(n)) + r4::kNoiseFloor;
    };
    auto store_y = [&](uint32_t t) __attribute__((always_inline)) {
      const float* b = y_slot(t);
      const v4f y0 = *reinterpret_cast<const v4f*>(b + 8 * c), y1 = *reinterpret_cast<const v4f*>(b + 8 * c + 4);
      const uint32_t tok = t * TT + c;
      if constexpr (EPI) {
        const v4f piece = r4::narrow(y0, y1);  // read.to(bf16)
        const v4f u[2] = {r4::widen_lo(piece), r4::widen_hi(piece)}, z[2] = {r4::widen_lo(xg), r4::widen_hi(xg)};
        float ss[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          ss[e] = u[e][0] * u[e][0];
#pragma unroll
          for (int k = 1; k < 4; ++k) ss[e] = fmaf(u[e][k], u[e][k], ss[e]);
        }
        const float r = __builtin_amdgcn_rsqf(fmaf(ss[0] + ss[1], 0.125f, a.norm_eps));
        v4f x[2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int k = 0; k < 4; ++k) x[e][k] = u[e][k] * r * a.norm_w[4 * e + k] * silu_(z[e][k]);
        const uint32_t off = tok * ro + head * 16u;
        if (precise) {
          r4::st128<r4::kNtStore>(rout, x[0], 2u * off, 0);
          r4::st128<r4::kNtStore>(rout, x[1], 2u * off + 16u, 0);
        } else {
          r4::st128<r4::kNtStore>(rout, r4::narrow(x[0], x[1]), off, 0);
        }
        r4::st128(ryb, piece, off, 0);
      } else {
        r4::st128<r4::kNtStore>(rout, y0, tok * yrow + head * 32u, 0);
        r4::st128<r4::kNtStore>(rout, y1, tok * yrow + head * 32u + 16u, 0);
      }
    };
    load(0);
    r4::vm_wait<0>();
    put(0);
    if (ntiles > 1) load(1);
    __syncthreads();
    for (uint32_t it = 0; it <= ntiles; ++it) {
      r4::vm_wait<0>();
      if (it + 1 < ntiles) put(it + 1);
      if (it >= 2) store_y(it - 2);
      if (it + 2 < ntiles) load(it + 2);
      if (it >= 1) load_gate(it - 1);
      __syncthreads();
    }
    r4::vm_wait<0>();
    store_y(ntiles - 1);
  }
}

// The streams wave's own pieces of the backward's chunks (a chunk is landed
// one step before its replay, and its gradients leave three steps after).
struct Raw {
  static constexpr int W = 6, SLOT = W * kWave, SIZE = SBTile::NSLOT * SLOT;
};

// G groups per workgroup: waves covariance reverse, mean, covariance replay
// and streams of each (with G = 2 the waves that share a SIMD are a reverse
// and a replay wave, a mean and a streams wave).
template <bool DYN, bool EPI, bool BIAS, int G>
__global__ __launch_bounds__(4 * G * kWave) void mixer_backward_row_kernel(MixArgs a) {
  __shared__ float lds_all[G * (SBTile::SIZE + Raw::SIZE)];
  constexpr int CH = SBTile::CH;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int role = wave / G, grp = wave % G;
  float* const lds = lds_all + grp * (SBTile::SIZE + Raw::SIZE);
  const int s = lane >> 4, c = lane & 15, i = c >> 2, j = c & 3;
  const float delta = i == j ? 1.f : 0.f;
  const Group g(a, static_cast<int64_t>(blockIdx.x) * G + grp);
  const uint32_t T = static_cast<uint32_t>(a.t);
  const uint32_t nbp = static_cast<uint32_t>(a.nb + 1);
  const int nb = static_cast<int>(a.nb);  // chunks; position x is chunk nb - 1 - x
  const int len0 = static_cast<int>(T) - (nb - 1) * CH;
  auto slot = [&](int x) __attribute__((always_inline)) {
    return lds + SBTile::IN + static_cast<int>(static_cast<uint32_t>(x) % SBTile::NSLOT) * SBTile::SLOT +
           s * SBTile::SEQ;
  };
  auto uslot = [&](int x) __attribute__((always_inline)) {
    return lds + SBTile::U + (x & 1) * SBTile::USLOT + s * SBTile::USEQ;
  };
  auto aslot = [&](int x) __attribute__((always_inline)) {
    return lds + SBTile::A + (x & 1) * SBTile::ASLOT + s * SBTile::ASEQ;
  };
  auto rslot = [&](int x) __attribute__((always_inline)) {
    return lds + SBTile::REC + static_cast<int>(static_cast<uint32_t>(x) % 3u) * SBTile::RSLOT + 4 * lane;
  };
  const uint32_t cvo = static_cast<uint32_t>(s) * 64u + cov_off(i, j);
  const uint32_t mo = static_cast<uint32_t>(s) * 128u + mean_off(i, j);
  // As backward_split_kernel: at step x the replay of chunk x, the mean of
  // chunk x - 1, the covariance reverse of chunk x - 2.
  if (role == 0) {
    const bool has_c = a.gcf != nullptr;
    const Rsrc rgc = make_rsrc(has_c ? a.gcf + g.n0 * 16 : a.c0, has_c ? g.valid * 64u : 0u);
    const uint32_t tr = static_cast<uint32_t>(s) * 64u + cov_off(j, i);
    float S = 0.5f * (r4::ld32(rgc, cvo, 0) + r4::ld32(rgc, tr, 0));
    First first = {0.f, 0.f, 0.f, 0.f, 0.f};
    __syncthreads();
    for (int x = 0; x <= nb + 1; ++x) {
      if (x >= 2) reverse_chunk<false, DYN>(S, first, slot(x - 2), aslot(x - 2), rslot(x - 2), i, j, delta, a.floor);
      __syncthreads();
    }
    if (a.gc0) {
      const Rsrc rgc0 = make_rsrc(a.gc0 + g.n0 * 16, g.valid * 64u);
      const float asym = 0.5f * (first.gui * first.kj - first.guj * first.ki);
      r4::st32(rgc0, fmaf(asym, first.dd, S), cvo, 0);
    }
  } else if (role == 1) {
    const bool has_m = a.gmf != nullptr;
    const Rsrc rgm = make_rsrc(has_m ? a.gmf + g.n0 * 32 : a.m0, has_m ? g.valid * 128u : 0u);
    const v2f m = ld64(rgm, mo, 0);
    float gM0 = m[0], gM1 = m[1];
    __syncthreads();
    for (int x = 0; x <= nb + 1; ++x) {
      if (x >= 1 && x <= nb) mean_chunk<false, DYN>(gM0, gM1, slot(x - 1), uslot(x - 1), aslot(x - 1), i, j, c);
      __syncthreads();
    }
    if (a.gm0) {
      const Rsrc rgm0 = make_rsrc(a.gm0 + g.n0 * 32, g.valid * 128u);
      v2f o;
      o[0] = gM0;
      o[1] = gM1;
      r4::st64(rgm0, o, mo, 0);
    }
  } else if (role == 2) {
    const Rsrc rbc = make_rsrc(a.bcr + g.n0 * nbp * 16, g.valid * nbp * 64u);
    const uint32_t cco = static_cast<uint32_t>(s) * nbp * 64u + cov_off(i, j);
    auto ckpt = [&](int x) __attribute__((always_inline)) {
      return r4::ld32(rbc, cco + static_cast<uint32_t>(nb - 1 - x) * 64u, 0);
    };
    float Pload = ckpt(0);
    __syncthreads();
    for (int x = 0; x <= nb + 1; ++x) {
      r4::vm_wait<0>();
      const float Pc = Pload;
      if (x + 1 < nb) Pload = ckpt(x + 1);
      if (x < nb) replay_chunk<false>(Pc, slot(x), uslot(x), rslot(x), i, j, delta, a.floor);
      __syncthreads();
    }
  } else {
    // Lane (s, c): token c & 7 of the chunk, head s, half c >> 3: k or q, four
    // of the values, two of the decays, process or observation noise.
    const int tk = c & 7, half = c >> 3;
    const bool hi = half != 0;
    const Rows rows(a, g);
    const r4::MixGrads gr(a, g.bb, g.h0);
    const uint32_t head = static_cast<uint32_t>(g.h0) + s;
    const uint32_t H = static_cast<uint32_t>(a.h), ro = H * 16u, yrow = H * 32u;
    const uint32_t rg = static_cast<uint32_t>(a.ldg * 2), rgg = static_cast<uint32_t>(a.ldgg ? a.ldgg : 8 * a.h) * 2u;
    const bool precise = a.precise != 0;
    const uint32_t on = g.valid ? T : 0u;
    const Rsrc rgate = make_rsrc(EPI ? as_f(a.gate, g.bb * a.t * rg) : a.m0, EPI ? on * rg : 0u);
    const Rsrc ryb = make_rsrc(EPI ? as_f(a.yb, g.bb * a.t * ro) : a.m0, EPI ? on * ro : 0u);
    const Rsrc rgo = EPI ? make_rsrc(as_f(a.gout, g.bb * a.t * ro), on * ro)
                         : make_rsrc(as_f(a.gy, g.bb * a.t * yrow), on * yrow);
    const uint32_t ggrow = precise ? 2u * rgg : rgg;
    const Rsrc rggate = make_rsrc(EPI ? as_f(a.ggate, g.bb * a.t * ggrow) : a.m0, EPI ? on * ggrow : 0u);
    const Rsrc rbm = make_rsrc(a.bmr + g.n0 * nbp * 32, g.valid * nbp * 128u);
    const uint32_t cmo = static_cast<uint32_t>(s) * nbp * 128u + mean_off(i, j);
    // Offsets of lanes that take no part (and of an empty group's stores).
    const uint32_t koff = hi ? kOob : head * 8u, qoff = hi ? head * 8u : kOob;
    const uint32_t voff = head * 16u + half * 8u, doff = head * 8u + half * 4u;
    uint32_t bd = 0, bn = 0;
    if constexpr (BIAS) {
      if (g.valid) {
        const uint32_t* ab = static_cast<const uint32_t*>(a.abias);
        bd = ab[2 * head + half];
        bn = ab[2 * H + head];
      }
    }
    float w[4], dw[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      w[k] = EPI ? a.norm_w[4 * half + k] : 0.f;
      dw[k] = 0.f;
    }
    v2f xk, xq, xv, xo, xy, xg, xm;
    v4f xgy;
    float xd, xn;
    auto load = [&](int x) __attribute__((always_inline)) {
      const uint32_t tok = static_cast<uint32_t>((nb - 1 - x) * CH + tk);
      xk = ld64(rows.k, hi ? kOob : tok * rows.rk + koff, 0);
      xq = ld64(rows.q, hi ? tok * rows.rq + qoff : kOob, 0);
      xv = ld64(rows.v, tok * rows.rv + voff, 0);
      xd = r4::ld32(rows.dl, tok * rows.rd + doff, 0);
      xn = r4::ld32(rows.nz, tok * rows.rn + head * 4u, 0);
      if constexpr (EPI) {
        xo = ld64(rgo, tok * ro + voff, 0);
        xy = ld64(ryb, tok * ro + voff, 0);
        xg = ld64(rgate, tok * rg + voff, 0);
      } else {
        xgy = r4::ld128<r4::kNtLoad>(rgo, tok * yrow + 2u * voff);
      }
      xm = ld64(rbm, cmo + static_cast<uint32_t>(nb - 1 - x) * 128u, 0);
    };
    auto raw = [&](int x) __attribute__((always_inline)) {
      return lds + SBTile::SIZE + static_cast<int>(static_cast<uint32_t>(x) % SBTile::NSLOT) * Raw::SLOT + lane;
    };
    auto put = [&](int x) __attribute__((always_inline)) {
      float* b = slot(x);
      float* keep = raw(x);
      const v2f kq = hi ? xq : xk;
      uint32_t d = word(xd), n = word(xn);
      if constexpr (BIAS) {
        d = add2(d, bd);
        n = add2(n, bn);
      }
      keep[0] = kq[0];
      keep[kWave] = kq[1];
      keep[2 * kWave] = xv[0];
      keep[3 * kWave] = xv[1];
      keep[4 * kWave] = __builtin_bit_cast(float, d);
      keep[5 * kWave] = __builtin_bit_cast(float, n);
      *reinterpret_cast<v4f*>(b + (hi ? SBTile::Q : SBTile::K) + 4 * tk) = r4::unit_silu(widen4(kq));
      const v4f v = widen4(xv);
      *reinterpret_cast<v4f*>(b + SBTile::V + 8 * tk + 4 * half) = silu4(v);
      v2f dd;
      dd[0] = r4::decay_(lo16(d));
      dd[1] = r4::decay_(hi16(d));
      *reinterpret_cast<v2f*>(b + SBTile::D + 4 * tk + 2 * half) = dd;
      b[(hi ? SBTile::R : SBTile::P) + tk] = r4::softplus_(hi ? hi16(n) : lo16(n)) + r4::kNoiseFloor;
      v4f gy;
      if constexpr (EPI) {
        // gy of the readout's epilogue, its gate gradient and weight-gradient
        // share (the equations of bssm_mixer.hip's put_epi; r = 0 for tokens
        // past T, as there).
        const v4f y = widen4(xy), z = widen4(xg), go = widen4(xo);
        float ss = y[0] * y[0];
#pragma unroll
        for (int k = 1; k < 4; ++k) ss = fmaf(y[k], y[k], ss);
        ss += dpp<kRowRor8>(ss);
        const float rms = __builtin_amdgcn_rsqf(fmaf(ss, 0.125f, a.norm_eps)), r = x == 0 && tk >= len0 ? 0.f : rms;
        v4f gz, gn, nn;
        float dot = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float sg = sigmoid_(z[k]), sz = z[k] * sg;
          const float dsz = fmaf(sz, -sg, sg + sz);
          nn[k] = y[k] * r;
          const float gh = go[k] * sz;
          gz[k] = go[k] * (nn[k] * w[k]) * dsz;
          gn[k] = gh * w[k];
          dw[k] = fmaf(gh, nn[k], dw[k]);
          dot = fmaf(gn[k], nn[k], dot);
        }
        dot += dpp<kRowRor8>(dot);
#pragma unroll
        for (int k = 0; k < 4; ++k) gy[k] = r * fmaf(-nn[k], dot * 0.125f, gn[k]);
        const uint32_t off = static_cast<uint32_t>((nb - 1 - x) * CH + tk) * rgg + voff;
        if (precise) r4::st128<r4::kNtStore>(rggate, gz, 2u * off, 0);
        else r4::st64(rggate, narrow4(gz), off, 0);
      } else {
        gy = xgy;
      }
      *reinterpret_cast<v4f*>(b + SBTile::GY + 8 * tk + 4 * half) = gy;
      *reinterpret_cast<v2f*>(b + SBTile::MC + 2 * c) = xm;
      if (x == 0 && len0 < CH) neutral_tail<SBTile, CH>(b, len0, c);
    };
    // Four (two) values of a gradient at the bf16 layout's byte offset.
    auto put4 = [&](Rsrc r, uint32_t off, v4f x) __attribute__((always_inline)) {
      if (gr.f32) r4::st128<r4::kNtStore>(r, x, off < kOob ? 2u * off : kOob, 0);
      else r4::st64(r, narrow4(x), off, 0);
    };
    auto put2 = [&](Rsrc r, uint32_t off, float x0, float x1) __attribute__((always_inline)) {
      if (gr.f32) {
        v2f x;
        x[0] = x0;
        x[1] = x1;
        r4::st64(r, x, off < kOob ? 2u * off : kOob, 0);
      } else {
        r4::st32(r, __builtin_bit_cast(float, narrow2(x0, x1)), off, 0);
      }
    };
    auto store = [&](int x) __attribute__((always_inline)) {
      const float* b = slot(x);
      const float* keep = raw(x);
      const uint32_t tok = static_cast<uint32_t>((nb - 1 - x) * CH + tk);
      v2f kq, xv;
      kq[0] = keep[0];
      kq[1] = keep[kWave];
      xv[0] = keep[2 * kWave];
      xv[1] = keep[3 * kWave];
      const v4f gt = *reinterpret_cast<const v4f*>(b + (hi ? SBTile::Q : SBTile::K) + 4 * tk);
      const v4f gkq = r4::unit_silu_grad(widen4(kq), gt);
      put4(gr.k, g.valid && !hi ? tok * gr.rk + head * 8u : kOob, gkq);
      put4(gr.q, g.valid && hi ? tok * gr.rq + head * 8u : kOob, gkq);
      const v4f z = widen4(xv), gvt = *reinterpret_cast<const v4f*>(b + SBTile::V + 8 * tk + 4 * half);
      v4f o;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float sg = sigmoid_(z[k]);
        o[k] = gvt[k] * sg * fmaf(z[k], 1.f - sg, 1.f);
      }
      put4(gr.v, g.valid ? tok * gr.rv + voff : kOob, o);
      if constexpr (DYN) {
        const uint32_t d = word(keep[4 * kWave]), n = word(keep[5 * kWave]);
        const v2f gd = *reinterpret_cast<const v2f*>(b + SBTile::D + 4 * tk + 2 * half);
        float od[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          // d/dz exp(-softplus(z)) = -sigmoid(|z|)^2 e^-|z|
          const float zz = k ? hi16(d) : lo16(d);
          const float ea = r4::exp_(-fabsf(zz)), sa = r4::rcp_(1.f + ea);
          od[k] = -gd[k] * (ea * sa) * sa;
        }
        put2(gr.dl, g.valid ? tok * gr.rd + doff : kOob, od[0], od[1]);
        const float gn = b[(hi ? SBTile::R : SBTile::P) + tk] * sigmoid_(hi ? hi16(n) : lo16(n));
        const float other = dpp<kRowRor8>(gn);
        put2(gr.nz, g.valid && !hi ? tok * gr.rn + head * 4u : kOob, gn, other);
      }
    };
    load(0);
    r4::vm_wait<0>();
    put(0);
    if (nb > 1) load(1);
    __syncthreads();
    for (int x = 0; x <= nb + 1; ++x) {
      r4::vm_wait<0>();
      if (x + 1 < nb) {
        put(x + 1);
        if (x + 2 < nb) load(x + 2);
      }
      if (x >= 3) store(x - 3);
      __syncthreads();
    }
    store(nb - 1);
    if constexpr (EPI) {
      // Rows of 8 partials, 4 for each 16 heads of a batch row (those past its
      // last head are zeros).
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        dw[k] += __shfl_xor(dw[k], 1);
        dw[k] += __shfl_xor(dw[k], 2);
        dw[k] += __shfl_xor(dw[k], 4);
        dw[k] += __shfl_xor(dw[k], 16);
        dw[k] += __shfl_xor(dw[k], 32);
      }
      if (g.valid) {
        const int64_t rows4 = (a.h + 15) / 16 * 4, mine = g.h0 / SPW;
        float* part = a.gw_part + (g.bb * rows4 + mine) * 8;
        if (tk == 0 && s == 0) {
#pragma unroll
          for (int k = 0; k < 4; ++k) part[4 * half + k] = dw[k];
        }
        if (g.h0 + SPW == a.h && lane < 8)
          for (int64_t r = 1; mine + r < rows4; ++r) part[8 * r + lane] = 0.f;
      }
    }
  }
}

// Groups up to which every workgroup of one group has a CU of its own.
constexpr int64_t kOneGroup = 256;

template <bool EPI, bool BIAS>
void launch_forward_row(const MixArgs& a, int64_t groups, hipStream_t stream) {
  if (groups > kOneGroup)
    hipLaunchKernelGGL((mixer_forward_row_kernel<EPI, BIAS, 2>), dim3(static_cast<unsigned>((groups + 1) / 2)),
                       dim3(6 * kWave), 0, stream, a);
  else
    hipLaunchKernelGGL((mixer_forward_row_kernel<EPI, BIAS, 1>), dim3(static_cast<unsigned>(groups)), dim3(3 * kWave),
                       0, stream, a);
}
template <bool DYN, bool EPI, bool BIAS>
void launch_backward_row(const MixArgs& a, int64_t groups, hipStream_t stream) {
  if (groups > kOneGroup)
    hipLaunchKernelGGL((mixer_backward_row_kernel<DYN, EPI, BIAS, 2>), dim3(static_cast<unsigned>((groups + 1) / 2)),
                       dim3(8 * kWave), 0, stream, a);
  else
    hipLaunchKernelGGL((mixer_backward_row_kernel<DYN, EPI, BIAS, 1>), dim3(static_cast<unsigned>(groups)),
                       dim3(4 * kWave), 0, stream, a);
}

}  // namespace
}  // namespace sn

hipError_t launch_mixer_forward_row(const MixArgs& a, hipStream_t stream) {
  const int64_t groups = a.b * (a.h / sn::SPW);
  if (groups == 0) return hipSuccess;
  if (a.gate != nullptr && a.abias != nullptr) sn::launch_forward_row<true, true>(a, groups, stream);
  else if (a.gate != nullptr) sn::launch_forward_row<true, false>(a, groups, stream);
  else sn::launch_forward_row<false, false>(a, groups, stream);
  return hipGetLastError();
}

hipError_t launch_mixer_backward_row(const MixArgs& a, hipStream_t stream) {
  const int64_t groups = a.b * (a.h / sn::SPW);
  if (groups == 0) return hipSuccess;
  const bool dyn = a.gdl != nullptr, epi = a.gate != nullptr;
  if (dyn && epi && a.abias != nullptr) sn::launch_backward_row<true, true, true>(a, groups, stream);
  else if (dyn && epi) sn::launch_backward_row<true, true, false>(a, groups, stream);
  else if (dyn) sn::launch_backward_row<true, false, false>(a, groups, stream);
  else if (epi) sn::launch_backward_row<false, true, false>(a, groups, stream);
  else sn::launch_backward_row<false, false, false>(a, groups, stream);
  return hipGetLastError();
}

}  // namespace bssm
