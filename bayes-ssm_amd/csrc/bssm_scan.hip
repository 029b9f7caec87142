// Static (A = I, Q = 0) associative scan in information form, gfx950.
//
// Equation reference: bayes_ssm/replay_ssm.py:251-270 and
// docs/associative_scan.md.  For every token t of batch row b:
//   L_t = inv(P0) + sum_{s<=t} k_s (k_s / r_s)^T
//   N_t = inv(P0) M0 + sum_{s<=t} (k_s / r_s) v_s^T
//   M_t = L_t^{-1} N_t (Cholesky),  y_t = M_t^T q_t
// and for the last token also P_T = L_T^{-1}.
//
// A workgroup of four waves takes 64 tokens of one batch row, lane = token:
//   1. three waves sum the prefix of the tokens before the 64 with matrix
//      instructions, the fourth inverts the prior;
//   2. every wave adds the prefix within the 64 tokens to it by a 64-lane DPP
//      scan per entry, and each lane factors its own token's L_t in registers
//      (no exchange between lanes, no LDS);
//   3. the value columns are split over the waves: a column's N_t comes of
//      the same scan, and each lane solves for its token.
// At 16 x 1000 tokens, D = M = 16, the forward takes 30 us and the backward
// 50 + 12 + 37 us; one wave per token that summed its whole prefix, with 16 of
// 64 lanes in the factorization and a suffix pass of one thread per entry, took
// 1400 and 1366 + 210 + 35 us.  (Step 1 on the VALU, lanes over the entries:
// 185 us forward.)  Bound by the instruction stream of a wave, one to a SIMD:
// 250 workgroups; step 1 grows with T^2 / 64.  Short sequences take a wave per
// token (short_sequences has the line).
//
// The key dimension is a template parameter (runtime D is padded up to the
// next instantiated size: the padded block of every matrix is the identity
// and the padded key entries are zero, which leaves the leading block of
// every factor and solution unchanged).  Instantiated for D = 1, 2, 4, 8, 16;
// larger key dimensions (up to 32) take the LDS kernel below.

#include "bssm_recurrence.h"

#include <type_traits>

namespace bssm {
namespace {

constexpr int kMaxD = 32;
constexpr int kMaxM = 64;
constexpr int kTok = 64;    // tokens per workgroup
constexpr int kWaves = 4;

// LDS written by some lanes of the wave is read by others after this (without
// it the compiler may read before the branch of the writing lanes is taken).
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Row-per-lane Cholesky: lane i < D holds row i of the SPD matrix A (lanes
// >= D hold zeros); on return it holds row i of the lower factor L (zeros
// above the diagonal) and inv_diag = 1 / L[i][i], and L is also in LDS
// (m, row-major) with its inverted diagonal in idg.  Each finished column is
// written to LDS, and column j reads the finished part of row j back with
// uniform addresses; only the pivot travels by readlane.
template <int D>
__device__ __forceinline__ void chol_rows(float (&a)[D], float& inv_diag, int lane, float* m, float* idg) {
#pragma unroll
  for (int j = 0; j < D; ++j) {
    float s = a[j];
#pragma unroll
    for (int k = 0; k < j; ++k) s = fmaf(-a[k], m[j * D + k], s);
    const float piv = sqrtf(__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, s), j)));
    const float rp = 1.0f / piv;
    a[j] = lane > j ? s * rp : (lane == j ? piv : 0.f);
    if (lane < D) m[lane * D + j] = a[j];
    if (lane == j) {
      inv_diag = rp;
      idg[j] = rp;
    }
    wave_fence();
  }
}

// Rows of a row-per-lane matrix into LDS (row-major, D x D), with the
// inverted diagonal of a factor in diag[] (only the first D lanes write).
template <int D>
__device__ __forceinline__ void rows_to_lds(const float (&a)[D], float* m, int lane) {
  if (lane < D) {
#pragma unroll
    for (int j = 0; j < D; j += 4) {
      v4f x;
      x[0] = a[j];
      x[1] = a[j + 1 < D ? j + 1 : j];
      x[2] = a[j + 2 < D ? j + 2 : j];
      x[3] = a[j + 3 < D ? j + 3 : j];
      if (j + 4 <= D) *reinterpret_cast<v4f*>(&m[lane * D + j]) = x;
      else
        for (int e = 0; e < D - j; ++e) m[lane * D + j + e] = x[e];
    }
  }
  wave_fence();
}

// Row i of an LDS matrix into registers (every lane reads the same words).
template <int D>
__device__ __forceinline__ void lds_row(const float* m, int i, float (&r)[D]) {
#pragma unroll
  for (int j = 0; j < D; j += 4) {
    if (j + 4 <= D) {
      const v4f x = *reinterpret_cast<const v4f*>(&m[i * D + j]);
      r[j] = x[0];
      r[j + 1] = x[1];
      r[j + 2] = x[2];
      r[j + 3] = x[3];
    } else {
      for (int e = 0; e < D - j; ++e) r[j + e] = m[i * D + j + e];
    }
  }
}

// Solve (L L^T) x = x in place for the calling lane's right-hand side; L
// (row-major) and 1 / diag(L) are in LDS and read with uniform addresses.
template <int D>
__device__ __forceinline__ void chol_solve(const float* L, const float* idg, float (&x)[D]) {
#pragma unroll
  for (int i = 0; i < D; ++i) {
    float li[D];
    lds_row<D>(L, i, li);
    float s = x[i];
#pragma unroll
    for (int k = 0; k < i; ++k) s = fmaf(-li[k], x[k], s);
    x[i] = s * idg[i];
  }
  // L^T x = z: column i of L is needed; rows k > i hold it at entry i.
#pragma unroll
  for (int i = D - 1; i >= 0; --i) {
    float s = x[i];
#pragma unroll
    for (int k = i + 1; k < D; ++k) s = fmaf(-L[k * D + i], x[k], s);
    x[i] = s * idg[i];
  }
}

// Padded (branch-free) element load: p[i] for i < n, else 0.
__device__ __forceinline__ float ld_or_zero(const float* p, int i, int n) {
  const float x = p[i < n ? i : 0];
  return i < n ? x : 0.f;
}

// Entries (i, j), j <= i, of a symmetric matrix in row order.
constexpr int tri(int i, int j) { return i * (i + 1) / 2 + j; }

// Inclusive sum over the lanes 0 .. l.
template <int CTRL, int ROWS, bool ZERO>
__device__ __forceinline__ float dpp_or_zero(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, ROWS, 0xF, ZERO));
}
__device__ __forceinline__ float lane_scan(float x) {
  x += dpp_or_zero<0x111, 0xF, true>(x);   // row_shr:1, 2, 4, 8: within rows of 16
  x += dpp_or_zero<0x112, 0xF, true>(x);
  x += dpp_or_zero<0x114, 0xF, true>(x);
  x += dpp_or_zero<0x118, 0xF, true>(x);
  x += dpp_or_zero<0x142, 0xA, false>(x);  // row_bcast:15 into rows 1 and 3
  return x + dpp_or_zero<0x143, 0xC, false>(x);  // row_bcast:31 into rows 2 and 3
}

// Sum over the lanes before l.  A token's own term is added to it by one fma:
// with a small r it is far larger than the rest, and rounded in each step of
// an inclusive scan it cost twice the error of the variances' gradient.
__device__ __forceinline__ float lane_scan_before(float x) {
  return lane_scan(dpp_or_zero<0x138, 0xF, true>(x));  // wave_shr:1
}

// Row-major rows of `cols` floats: entries 4 u .. 4 u + 3 of a row (zero past
// n).  VEC: n is a multiple of 4 (rows need 4-byte alignment only).
template <bool VEC>
__device__ __forceinline__ v4f row4(const float* row, int u, int n) {
  if constexpr (VEC) return *reinterpret_cast<const v4f_a4*>(row + 4 * u);
  v4f x;
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = ld_or_zero(row, 4 * u + e, n);
  return x;
}

template <int D>
struct Lds {
  static constexpr int KP = D < 4 ? 4 : D;                       // padded key columns
  static constexpr int kCols = 16 + kMaxM;  // row i of the prefix sums: k_i / r times k, at 16 times v
  float part[3][D * kCols];                 // of three waves
  float base[D * KP];        // inv(P0) + prefix before the workgroup's tokens (symmetric)
  float nbase[kMaxM * KP];   // the same for N, one value column after the other
  float mat[D * D];          // a factor or inv(P0), row-major
  float idg[D];              // 1 / diag of the factor in mat
};

struct ScanIn {
  const float *k, *v, *q, *r, *m0, *c0;
  int64_t T;
  int d, m;
};

// Step 1: base and nbase of the workgroup's tokens (first token t0).
template <int D, bool VEC>
__device__ __forceinline__ void prefix_base(const ScanIn& a, int64_t b, int64_t t0, int wave, int lane, Lds<D>& l) {
  constexpr int KP = Lds<D>::KP, kCols = Lds<D>::kCols;
  const int Dr = VEC ? D : a.d, M = a.m;
  if (wave < 3) {
    // (k / r)^T [k v] over the tokens before t0 (a multiple of 64), four to a
    // matrix instruction: operand lane = token 4 s + lane / 16, row or column
    // lane % 16.  A wave's batch of eight has its loads in flight together.
    const int col = lane & 15;
    v4f acc[1 + kMaxM / 16];
#pragma unroll
    for (int n = 0; n <= kMaxM / 16; ++n) acc[n] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int64_t s = wave * 32; s < t0; s += 3 * 32) {
      const int64_t tok = b * a.T + s + lane / 16;
      float kx[8], wx[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        kx[u] = ld_or_zero(a.k + (tok + 4 * u) * Dr, col, Dr);
        wx[u] = a.r[tok + 4 * u];
      }
#pragma unroll
      for (int n = 0; n < kMaxM / 16; ++n) {
        if (16 * n < M) {
          float vx[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) vx[u] = ld_or_zero(a.v + (tok + 4 * u) * M, 16 * n + col, M);
          if (n == 0) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              wx[u] = kx[u] * (1.0f / wx[u]);
              acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(wx[u], kx[u], acc[0], 0, 0, 0);
            }
          }
#pragma unroll
          for (int u = 0; u < 8; ++u)
            acc[1 + n] = __builtin_amdgcn_mfma_f32_16x16x4f32(wx[u], vx[u], acc[1 + n], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int n = 0; n <= kMaxM / 16; ++n) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 4 * (lane / 16) + e;
        if (row < D && 16 * (n - 1) < M) l.part[wave][row * kCols + 16 * n + col] = acc[n][e];
      }
    }
  } else {
    // inv(P0): factor P0 (padded with the identity), then lane c < D solves
    // for column c of the identity; column c of inv(P0) is its row c.
    const bool row_lane = lane < Dr, col_lane = lane < M;
    float f[D], inv_diag = 1.f, lam0[D];
    const float* P0 = a.c0 + (b * Dr + (row_lane ? lane : 0)) * Dr;
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const float v = ld_or_zero(P0, j, Dr);
      f[j] = row_lane ? v : (lane == j ? 1.f : 0.f);
    }
    float m0c[D];
    const float* M0 = a.m0 + b * Dr * M + (col_lane ? lane : 0);
#pragma unroll
    for (int k = 0; k < D; ++k) {
      const float v = M0[(k < Dr ? k : 0) * M];
      m0c[k] = (col_lane && k < Dr) ? v : 0.f;
    }
    chol_rows<D>(f, inv_diag, lane, l.mat, l.idg);
#pragma unroll
    for (int j = 0; j < D; ++j) lam0[j] = lane == j ? 1.f : 0.f;
    chol_solve<D>(l.mat, l.idg, lam0);
    rows_to_lds<D>(lam0, l.mat, lane);  // mat = inv(P0)
    // N_t column c starts at inv(P0) M0[:, c].
#pragma unroll
    for (int i = 0; i < D; ++i) {
      float li[D];
      lds_row<D>(l.mat, i, li);
      float n0 = 0.f;
#pragma unroll
      for (int k = 0; k < D; ++k) n0 = fmaf(li[k], m0c[k], n0);
      if (col_lane) l.nbase[lane * KP + i] = n0;
    }
  }
  __syncthreads();
  const int tid = wave * kWave + lane;
  auto sum3 = [&](int e) __attribute__((always_inline)) { return (l.part[0][e] + l.part[1][e]) + l.part[2][e]; };
  for (int e = tid; e < D * D; e += kWaves * kWave) {
    const int i = e / D, j = e - i * D;
    const float s0 = 0.5f * (l.mat[i * D + j] + l.mat[j * D + i]);
    l.base[i * KP + j] = s0 + 0.5f * (sum3(i * kCols + j) + sum3(j * kCols + i));
  }
  for (int e = tid; e < D * M; e += kWaves * kWave) {
    const int c = e / D, i = e - c * D;
    l.nbase[c * KP + i] += sum3(i * kCols + 16 + c);
  }
  __syncthreads();
}

// The lane's token.
template <int D>
struct Tok {
  float k[D], wk[D];          // k and k / r (zero past T)
  float L[D * (D + 1) / 2];   // factor of L_t, the diagonal inverted
};

// Solve L x = b, then L^T x = b, in place.
template <int D>
__device__ __forceinline__ void solve(const float (&L)[D * (D + 1) / 2], float (&x)[D]) {
#pragma unroll
  for (int i = 0; i < D; ++i) {
    float s = x[i];
#pragma unroll
    for (int k = 0; k < i; ++k) s = fmaf(-L[tri(i, k)], x[k], s);
    x[i] = s * L[tri(i, i)];
  }
#pragma unroll
  for (int i = D - 1; i >= 0; --i) {
    float s = x[i];
#pragma unroll
    for (int k = i + 1; k < D; ++k) s = fmaf(-L[tri(k, i)], x[k], s);
    x[i] = s * L[tri(i, i)];
  }
}

// The token's key, precision (base + scan) and factor.
template <int D, bool VEC>
__device__ __forceinline__ void factor_token(const ScanIn& a, int64_t b, int64_t t0, int lane, const Lds<D>& l,
                                             Tok<D>& x) {
  constexpr int KP = Lds<D>::KP;
  const int Dr = VEC ? D : a.d;
  const bool valid = t0 + lane < a.T;
  const int64_t t = b * a.T + (valid ? t0 + lane : 0);
  const float rinv = 1.0f / a.r[t];
#pragma unroll
  for (int u = 0; u < KP / 4; ++u) {
    const v4f kv = row4<VEC>(a.k + t * Dr, u, Dr);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (4 * u + e < D) {
        x.k[4 * u + e] = valid ? kv[e] : 0.f;
        x.wk[4 * u + e] = valid ? kv[e] * rinv : 0.f;
      }
  }
#pragma unroll
  for (int i = 0; i < D; ++i) {
#pragma unroll
    for (int j = 0; j <= i; ++j) x.L[tri(i, j)] = fmaf(x.wk[i], x.k[j], l.base[i * KP + j] + lane_scan_before(x.wk[i] * x.k[j]));
  }
#pragma unroll
  for (int j = 0; j < D; ++j) {
    float s = x.L[tri(j, j)];
#pragma unroll
    for (int k = 0; k < j; ++k) s = fmaf(-x.L[tri(j, k)], x.L[tri(j, k)], s);
    const float rp = 1.0f / sqrtf(s);
    x.L[tri(j, j)] = rp;
#pragma unroll
    for (int i = j + 1; i < D; ++i) {
      float z = x.L[tri(i, j)];
#pragma unroll
      for (int k = 0; k < j; ++k) z = fmaf(-x.L[tri(i, k)], x.L[tri(j, k)], z);
      x.L[tri(i, j)] = z * rp;
    }
  }
}

// Column c of the token's mean M_t = L_t^{-1} N_t.
template <int D>
__device__ __forceinline__ void mean_column(const Tok<D>& x, const Lds<D>& l, int c, float vc, float (&mc)[D]) {
  constexpr int KP = Lds<D>::KP;
#pragma unroll
  for (int i = 0; i < D; ++i) mc[i] = fmaf(x.wk[i], vc, l.nbase[c * KP + i] + lane_scan_before(x.wk[i] * vc));
  solve<D>(x.L, mc);
}

// The factor held by lane `src` into l.mat (row-major, lower) and l.idg.
template <int D>
__device__ __forceinline__ void factor_to_lds(const Tok<D>& x, int lane, int src, Lds<D>& l) {
  if (lane == src) {
#pragma unroll
    for (int i = 0; i < D; ++i) {
#pragma unroll
      for (int j = 0; j < i; ++j) l.mat[i * D + j] = x.L[tri(i, j)];
      l.idg[i] = x.L[tri(i, i)];
    }
  }
  wave_fence();
}

template <int D, bool VEC>
__global__ __launch_bounds__(kWaves* kWave) void scan_forward_kernel(ScanIn a, float* __restrict__ out,
                                                                    float* __restrict__ mT, float* __restrict__ cT) {
  __shared__ Lds<D> l;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int Dr = VEC ? D : a.d, M = a.m;
  const int64_t b = blockIdx.y, t0 = static_cast<int64_t>(blockIdx.x) * kTok;
  prefix_base<D, VEC>(a, b, t0, wave, lane, l);
  Tok<D> x;
  factor_token<D, VEC>(a, b, t0, lane, l, x);
  const bool valid = t0 + lane < a.T;
  const int64_t t = b * a.T + (valid ? t0 + lane : 0);
  float q[D];
#pragma unroll
  for (int i = 0; i < D; ++i) q[i] = ld_or_zero(a.q + t * Dr, i, Dr);
  const bool last = t0 + lane == a.T - 1;
  for (int c = wave; c < M; c += kWaves) {
    const float vv = a.v[t * M + c];
    float mc[D];
    mean_column<D>(x, l, c, valid ? vv : 0.f, mc);
    float y = 0.f;
#pragma unroll
    for (int i = 0; i < D; ++i) y = fmaf(mc[i], q[i], y);
    if (valid) out[t * M + c] = y;
    if (last) {
#pragma unroll
      for (int i = 0; i < D; ++i)
        if (i < Dr) mT[(b * Dr + i) * M + c] = mc[i];
    }
  }
  if (t0 + kTok >= a.T && wave == 0) {
    // P_T = L_T^{-1}: lane c solves for column c of the identity.  (The other
    // waves have read mat before the barriers of prefix_base.)
    factor_to_lds<D>(x, lane, static_cast<int>(a.T - 1 - t0), l);
    float e[D];
#pragma unroll
    for (int i = 0; i < D; ++i) e[i] = lane == i ? 1.f : 0.f;
    chol_solve<D>(l.mat, l.idg, e);
    if (lane < Dr) {
#pragma unroll
      for (int i = 0; i < D; ++i)
        if (i < Dr) cT[(b * Dr + i) * Dr + lane] = e[i];
    }
  }
}

// ------------------------------------------------------------------ backward
// Reverse of the scan (the chain rule of replay_ssm.py:251-270).  With
// G_t = q_t gy_t^T (+ gM_T at the last token) the adjoint of M_t:
//   gq_t = M_t gy_t,   gN_t = L_t^{-1} G_t,
//   gL_t = sym(-gN_t M_t^T)  (+ sym(-P_T gP_T P_T) at the last token),
// where sym is the symmetrization the forward applies to L_t.  With the
// suffix sums SL_s = sum_{t>=s} gL_t and SN_s = sum_{t>=s} gN_t of the
// prefix terms k_s k_s^T / r_s and k_s v_s^T / r_s:
//   gk_s = (2 SL_s k_s + SN_s v_s) / r_s,   gv_s = SN_s^T k_s / r_s,
//   gr_s = -(k_s^T SL_s k_s + k_s^T SN_s v_s) / r_s^2,
// and for the prior (L_0 = inv(P0), N_0 = inv(P0) M0):
//   gM0 = inv(P0) SN_0,   gP0 = -inv(P0)^T (SL_0 + SN_0 M0^T) inv(P0)^T.
// Pass 1 (the forward's workgroups) writes gq, and gL_t (lower triangle) and
// gN_t into the workspace, entry by entry with a workgroup's tokens side by
// side; pass 2 turns each entry's 64 tokens into their suffix sums (one wave
// an entry, a lane scan); pass 3 (a workgroup per 64 tokens, lane = token)
// adds the sums of the later tokens' blocks, which stand at their first
// tokens, and forms the gradients; its first workgroup also the prior's.
struct Ws {
  float* p;
  int64_t T;
  int d, m;
  // Entry e (gL's triangle, then gN row by row) of the block of tokens at t0,
  // and the number of tokens in it.
  __device__ __forceinline__ int len(int64_t t0) const {
    return static_cast<int>(T - t0 < kTok ? T - t0 : kTok);
  }
  __device__ __forceinline__ float* at(int64_t b, int64_t t0, int e) const {
    return p + (b * T + t0) * (d * d + d * m) + static_cast<int64_t>(e) * len(t0);
  }
};
//
// k^T SL k and k^T SN v cancel where r is small (M^T k is then near v), so
// that single roundings of gL and of the sums show in gr: gL is summed over
// the columns, the suffixes over the tokens and gk and gr over the rows in
// float64 (at the rate of float32 here) and rounded where they are stored.

// Row m of the rows of gL that wave W sums (their lengths add up to the same
// for every wave at D = 8 and 16).
template <int D, int W>
constexpr int gl_row(int m) {
  return D <= 4 ? (m == 0 && W < D ? W : D) : (m & 1 ? 4 * m + 3 - W : 4 * m + W);
}

template <int D, int W>
struct GlRows {
  static constexpr int kRows = D <= 4 ? 1 : D / 4;
  double acc[kRows][D];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int m = 0; m < kRows; ++m)
#pragma unroll
      for (int j = 0; j < D; ++j) acc[m][j] = 0.;
  }
  // Column: mean in x[0 .. D), gN in x[D .. 2 D), lane apart kWave.
  __device__ __forceinline__ void add(const float* x) {
    double mc[D], g[D];
#pragma unroll
    for (int i = 0; i < D; ++i) {
      mc[i] = x[i * kWave];
      g[i] = x[(D + i) * kWave];
    }
#pragma unroll
    for (int m = 0; m < kRows; ++m) {
      constexpr auto row = gl_row<D, W>;
#pragma unroll
      for (int j = 0; j < D; ++j)
        if (row(m) < D && j <= row(m))
          acc[m][j] = fma(-g[row(m) % D], mc[j], fma(-g[j], mc[row(m) % D], acc[m][j]));
    }
  }
};

template <int D, bool VEC>
__global__ __launch_bounds__(kWaves* kWave) void scan_backward_token_kernel(ScanIn a, const float* __restrict__ gy,
                                                                           const float* __restrict__ gmT,
                                                                           const float* __restrict__ gcT, Ws ws,
                                                                           float* __restrict__ gq) {
  __shared__ Lds<D> l;
  __shared__ float xch[2][kWaves][2 * D][kWave];  // a round's columns of the mean and gN
  __shared__ float pt[D * D], pgp[D * D];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int Dr = VEC ? D : a.d, M = a.m;
  const int64_t b = blockIdx.y, t0 = static_cast<int64_t>(blockIdx.x) * kTok;
  prefix_base<D, VEC>(a, b, t0, wave, lane, l);
  Tok<D> x;
  factor_token<D, VEC>(a, b, t0, lane, l, x);
  const bool valid = t0 + lane < a.T, last = t0 + lane == a.T - 1;
  const int64_t t = b * a.T + (valid ? t0 + lane : 0);
  const bool final_cov = gcT != nullptr && t0 + kTok >= a.T;
  if (final_cov && wave == 0) {
    // P_T gP_T P_T (row owners), with P_T from the last token's factor.
    factor_to_lds<D>(x, lane, static_cast<int>(a.T - 1 - t0), l);
    float e[D];
#pragma unroll
    for (int i = 0; i < D; ++i) e[i] = lane == i ? 1.f : 0.f;
    chol_solve<D>(l.mat, l.idg, e);  // lane c < D: column c of P_T (= row c)
    rows_to_lds<D>(e, pt, lane);
    float ar[D], pr[D];
#pragma unroll
    for (int j = 0; j < D; ++j) {
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < D; ++k) {
        const float gkj = (k < Dr && j < Dr) ? gcT[(b * Dr + k) * Dr + j] : 0.f;
        acc = fmaf(e[k], gkj, acc);
      }
      ar[j] = acc;
    }
#pragma unroll
    for (int j = 0; j < D; ++j) {
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < D; ++k) acc = fmaf(ar[k], pt[k * D + j], acc);
      pr[j] = acc;
    }
    rows_to_lds<D>(pr, pgp, lane);
  }
  float q[D], gqa[D];
#pragma unroll
  for (int i = 0; i < D; ++i) {
    q[i] = ld_or_zero(a.q + t * Dr, i, Dr);
    gqa[i] = 0.f;
  }
  const int tri_r = Dr * (Dr + 1) / 2;
  auto columns = [&](auto which) __attribute__((always_inline)) {
    constexpr int W = decltype(which)::value;
    GlRows<D, W> gl;
    gl.clear();
    int buf = 0;
    for (int c0 = 0; c0 < M; c0 += kWaves, buf ^= 1) {
      const int c = c0 + W;
      if (c < M) {
        const float vv = a.v[t * M + c], gg = gy[t * M + c];
        const float gyc = valid ? gg : 0.f;
        float mc[D], g[D];
        mean_column<D>(x, l, c, valid ? vv : 0.f, mc);
#pragma unroll
        for (int i = 0; i < D; ++i) {
          g[i] = q[i] * gyc;
          if (gmT != nullptr && i < Dr) {
            const float gm = gmT[(b * Dr + i) * M + c];
            g[i] = last ? g[i] + gm : g[i];
          }
        }
        solve<D>(x.L, g);  // gN_t, column c
#pragma unroll
        for (int i = 0; i < D; ++i) {
          gqa[i] = fmaf(mc[i], gyc, gqa[i]);
          if (i < Dr && valid) ws.at(b, t0, tri_r + i * M + c)[lane] = g[i];
          xch[buf][W][i][lane] = mc[i];
          xch[buf][W][D + i][lane] = g[i];
        }
      }
      // The buffer is written again two rounds on, behind the next barrier.
      __syncthreads();
      const int n = M - c0 < kWaves ? M - c0 : kWaves;
      for (int w = 0; w < n; ++w) gl.add(&xch[buf][w][0][lane]);
    }
#pragma unroll
    for (int m = 0; m < GlRows<D, W>::kRows; ++m) {
      constexpr auto row = gl_row<D, W>;
#pragma unroll
      for (int j = 0; j < D; ++j) {
        if (row(m) < D && j <= row(m) && row(m) < Dr && valid) {
          const int i = row(m) % D;
          // gL summed g mc^T + mc g^T: half of it is sym(g mc^T).
          double s = 0.5 * gl.acc[m][j];
          if (final_cov && last) s -= 0.5 * (static_cast<double>(pgp[i * D + j]) + pgp[j * D + i]);
          ws.at(b, t0, tri(i, j))[lane] = static_cast<float>(s);
        }
      }
    }
  };
  if (wave == 0) columns(std::integral_constant<int, 0>{});
  else if (wave == 1) columns(std::integral_constant<int, 1>{});
  else if (wave == 2) columns(std::integral_constant<int, 2>{});
  else columns(std::integral_constant<int, 3>{});
  __syncthreads();
  // gq: the waves' columns added up.
#pragma unroll
  for (int i = 0; i < D; ++i) xch[0][wave][i][lane] = gqa[i];
  __syncthreads();
  if (valid) {
    for (int i = wave; i < Dr; i += kWaves)
      gq[t * Dr + i] = (xch[0][0][i][lane] + xch[0][1][i][lane]) + (xch[0][2][i][lane] + xch[0][3][i][lane]);
  }
}

// Inclusive sum over the lanes 0 .. l.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_step(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(u), CTRL, ROWS, 0xF, ROWS == 0xF);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(u >> 32), CTRL, ROWS, 0xF, ROWS == 0xF);
  return x + __builtin_bit_cast(double, static_cast<uint64_t>(hi) << 32 | lo);
}
__device__ __forceinline__ double lane_scan64(double x) {
  x = dpp_step<0x118, 0xF>(dpp_step<0x114, 0xF>(dpp_step<0x112, 0xF>(dpp_step<0x111, 0xF>(x))));
  return dpp_step<0x143, 0xC>(dpp_step<0x142, 0xA>(x));
}

// Pass 2: the suffix sums over a block's tokens of kPass2 entries per wave.
constexpr int kPass2 = 8;
__global__ __launch_bounds__(kWaves* kWave) void scan_backward_suffix_kernel(Ws ws, int entries) {
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int64_t b = blockIdx.y, t0 = static_cast<int64_t>(blockIdx.x) * kTok;
  const int len = ws.len(t0);
  const int e0 = (blockIdx.z * kWaves + wave) * kPass2;
  float x[kPass2];
#pragma unroll
  for (int i = 0; i < kPass2; ++i) {
    const bool mine = lane < len && e0 + i < entries;
    x[i] = mine ? ws.at(b, t0, e0 + i)[len - 1 - lane] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < kPass2; ++i) x[i] = static_cast<float>(lane_scan64(x[i]));
#pragma unroll
  for (int i = 0; i < kPass2; ++i)
    if (lane < len && e0 + i < entries) ws.at(b, t0, e0 + i)[len - 1 - lane] = x[i];
}

// The prior's gradients: SL_0 (lane i < D: row i), SN_0 (lane c < M: column c;
// also row-major in sn), inv(P0) again (as in the forward), then gM0 = inv(P0)
// SN_0 and gP0 = -inv(P0)^T (SL_0 + SN_0 M0^T) inv(P0)^T.  One wave; mat, idg and
// tmp ([D][D]) are its LDS.
template <int D>
__device__ __forceinline__ void prior_grads(const ScanIn& a, int64_t b, int Dr, int lane, const float (&sl)[D],
                                            const float (&snc)[D], const float* sn, float* mat, float* idg,
                                            float* tmp, float* __restrict__ gm0, float* __restrict__ gc0) {
  const int M = a.m;
  const bool row_lane = lane < Dr, col_lane = lane < M;
  const int rl = row_lane ? lane : 0;
  float f[D], inv_diag = 1.f;
  const float* P0 = a.c0 + (b * Dr + rl) * Dr;
#pragma unroll
  for (int j = 0; j < D; ++j) {
    const float v = ld_or_zero(P0, j, Dr);
    f[j] = row_lane ? v : (lane == j ? 1.f : 0.f);
  }
  chol_rows<D>(f, inv_diag, lane, mat, idg);
  float lam0[D];
#pragma unroll
  for (int j = 0; j < D; ++j) lam0[j] = lane == j ? 1.f : 0.f;
  chol_solve<D>(mat, idg, lam0);  // lane i < D: column i of inv(P0)
  rows_to_lds<D>(lam0, mat, lane);  // mat = inv(P0)^T, row i = column i of inv(P0)
  if (col_lane) {
    // gM0[i][c] = sum_k inv(P0)[i][k] SN[k][c]
#pragma unroll
    for (int i = 0; i < D; ++i) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < D; ++j) s = fmaf(mat[j * D + i], snc[j], s);
      if (i < Dr) gm0[(b * Dr + i) * M + lane] = s;
    }
  }
  // gA = SL_0 + SN_0 M0^T (row owners, row i), then gP0 = -inv(P0)^T gA inv(P0)^T.
  float ga[D];
  const float* M0 = a.m0 + b * Dr * M;
#pragma unroll
  for (int j = 0; j < D; ++j) {
    float s = sl[j];
    if (row_lane && j < Dr)
      for (int c = 0; c < M; ++c) s = fmaf(sn[lane * kMaxM + c], M0[j * M + c], s);
    ga[j] = s;
  }
  float ta[D];
#pragma unroll
  for (int j = 0; j < D; ++j) {
    // (gA inv(P0)^T)[i][j] = sum_k gA[i][k] inv(P0)[j][k]
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < D; ++i) s = fmaf(ga[i], mat[i * D + j], s);
    ta[j] = s;
  }
  if (lane < D) {
#pragma unroll
    for (int j = 0; j < D; ++j) tmp[lane * D + j] = ta[j];
  }
  wave_fence();
  if (row_lane) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      // gP0[i][j] = -sum_k inv(P0)[k][i] (gA inv(P0)^T)[k][j]
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < D; ++i) s = fmaf(mat[lane * D + i], tmp[i * D + j], s);
      if (j < Dr) gc0[(b * Dr + lane) * Dr + j] = -s;
    }
  }
}

template <int D, bool VEC>
__global__ __launch_bounds__(kWaves* kWave) void scan_backward_input_kernel(ScanIn a, Ws ws, float* __restrict__ gk,
                                                                           float* __restrict__ gv,
                                                                           float* __restrict__ gr,
                                                                           float* __restrict__ gm0,
                                                                           float* __restrict__ gc0) {
  constexpr int TRI = D * (D + 1) / 2;
  __shared__ double carry[TRI + D * kMaxM];  // sums of the later blocks, per entry
  __shared__ double red[kWaves][2 * D][kWave], zsum[kWaves][kWave];
  __shared__ float mat[D * D], idg[D], sn[D * kMaxM];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int Dr = VEC ? D : a.d, M = a.m, tri_r = Dr * (Dr + 1) / 2, entries = tri_r + Dr * M;
  const int64_t b = blockIdx.y, t0 = static_cast<int64_t>(blockIdx.x) * kTok;
  for (int e = threadIdx.x; e < entries; e += kWaves * kWave) {
    double s = 0.;
#pragma unroll 4
    for (int64_t u = (a.T - 1) / kTok * kTok; u > t0; u -= kTok) s += *ws.at(b, u, e);
    carry[e] = s;
  }
  __syncthreads();
  const bool valid = t0 + lane < a.T;
  const int64_t t = b * a.T + (valid ? t0 + lane : 0);
  const int at = valid ? lane : 0;
  const float rinv = 1.0f / a.r[t];
  // Rows of SL k and SN v over the wave's rows and columns.
  double k[D], sk[D], nv[D];
#pragma unroll
  for (int i = 0; i < D; ++i) {
    k[i] = ld_or_zero(a.k + t * Dr, i, Dr);
    sk[i] = nv[i] = 0.;
  }
#pragma unroll
  for (int i = 0; i < D; ++i) {
    if ((i & (kWaves - 1)) == wave && i < Dr) {
#pragma unroll
      for (int j = 0; j <= i; ++j) {
        const double s = ws.at(b, t0, tri(i, j))[at] + carry[tri(i, j)];
        sk[i] = fma(s, k[j], sk[i]);
        if (j < i) sk[j] = fma(s, k[i], sk[j]);
      }
    }
  }
  for (int c = wave; c < M; c += kWaves) {
    const double vc = a.v[t * M + c];
    double acc = 0.;
#pragma unroll
    for (int i = 0; i < D; ++i) {
      if (i < Dr) {
        const int e = tri_r + i * M + c;
        const double s = ws.at(b, t0, e)[at] + carry[e];
        nv[i] = fma(s, vc, nv[i]);
        acc = fma(s, k[i], acc);
      }
    }
    if (valid) gv[t * M + c] = static_cast<float>(acc) * rinv;
  }
#pragma unroll
  for (int i = 0; i < D; ++i) {
    red[wave][i][lane] = sk[i];
    red[wave][D + i][lane] = nv[i];
  }
  __syncthreads();
  double z = 0.;
#pragma unroll
  for (int i = 0; i < D; ++i) {
    if ((i & (kWaves - 1)) == wave) {
      auto sum4 = [&](int e) __attribute__((always_inline)) {
        return (red[0][e][lane] + red[1][e][lane]) + (red[2][e][lane] + red[3][e][lane]);
      };
      const double x = sum4(i), y = sum4(D + i);
      z = fma(x + y, k[i], z);
      if (i < Dr && valid) gk[t * Dr + i] = static_cast<float>(2. * x + y) * rinv;
    }
  }
  zsum[wave][lane] = z;
  __syncthreads();
  if (wave == 0 && valid)
    gr[t] = -static_cast<float>((zsum[0][lane] + zsum[1][lane]) + (zsum[2][lane] + zsum[3][lane])) * rinv * rinv;
  if (t0 != 0 || wave != 0) return;
  const bool row_lane = lane < Dr, col_lane = lane < M;
  const int rl = row_lane ? lane : 0;
  float sl[D], snc[D];
#pragma unroll
  for (int j = 0; j < D; ++j) {
    const int jj = j < Dr ? j : 0;
    const int e = rl >= jj ? tri(rl, jj) : tri(jj, rl), en = tri_r + jj * M + (col_lane ? lane : 0);
    const float s = *ws.at(b, 0, e) + static_cast<float>(carry[e]), n = *ws.at(b, 0, en) + static_cast<float>(carry[en]);
    sl[j] = (row_lane && j < Dr) ? s : 0.f;
    snc[j] = (col_lane && j < Dr) ? n : 0.f;
  }
  if (col_lane) {
#pragma unroll
    for (int i = 0; i < D; ++i) sn[i * kMaxM + lane] = snc[i];
  }
  wave_fence();
  // tmp takes the place of carry, which no other wave reads now.
  prior_grads<D>(a, b, Dr, lane, sl, snc, sn, mat, idg, reinterpret_cast<float*>(carry), gm0, gc0);
}

// ------------------------------------------------------- short sequences
// One wave per (b, t): a workgroup of 64 tokens takes the time of 64 whatever
// part of them its row has.  Two lane roles: row owners (lane i < D) hold row i
// of the precision, then of its factor; column owners (lane c < M) hold column c
// of the natural parameter and solve for column c of the mean.  The prefix is
// summed token by token (rows s are uniform across the wave and load as scalars),
// eight to a partial sum.  EXACT: the key dimension equals D.  At D = M = 16 a
// batch of 2048 rows of 8 tokens takes 322 us backward, against 484 us with a
// workgroup per 64 tokens; 8192 of one token, forward and backward through the
// API, 381 against 2612 us.
// On return LDS mat / idg hold the factor of L_t and 1 / its diagonal, and the
// column owners column c of M_t = L_t^{-1} N_t in x.
template <int D, bool EXACT>
__device__ __forceinline__ void token_state(const ScanIn& a, int64_t b, int64_t t, int lane, float* mat, float* tr,
                                            float* idg, float (&x)[D]) {
  const int Dr = EXACT ? D : a.d, M = a.m;
  const bool row_lane = lane < Dr, col_lane = lane < M;
  const int rl = row_lane ? lane : 0, cl = col_lane ? lane : 0;
  // inv(P0): factor P0 (padded with the identity), then lane c < D solves for
  // column c of the identity; column c of inv(P0) is its row c (symmetric).
  float l[D], inv_diag = 1.f, lam0[D];
  const float* P0 = a.c0 + (b * Dr + rl) * Dr;
#pragma unroll
  for (int j = 0; j < D; ++j) {
    const float v = ld_or_zero(P0, j, Dr);
    l[j] = row_lane ? v : (lane == j ? 1.f : 0.f);
  }
  chol_rows<D>(l, inv_diag, lane, mat, idg);
#pragma unroll
  for (int j = 0; j < D; ++j) lam0[j] = lane == j ? 1.f : 0.f;
  chol_solve<D>(mat, idg, lam0);
  wave_fence();
  rows_to_lds<D>(lam0, mat, lane);  // mat = inv(P0)
  // N_t column c starts at inv(P0) M0[:, c].
  float m0c[D];
  const float* M0 = a.m0 + b * Dr * M + cl;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const float v = M0[(k < Dr ? k : 0) * M];
    m0c[k] = (col_lane && k < Dr) ? v : 0.f;
  }
#pragma unroll
  for (int i = 0; i < D; ++i) {
    float li[D];
    lds_row<D>(mat, i, li);
    float n0 = 0.f;
#pragma unroll
    for (int k = 0; k < D; ++k) n0 = fmaf(li[k], m0c[k], n0);
    x[i] = n0;
  }
  // Prefix sums over s < t: row owners row i of sum k (k / r)^T, column
  // owners column c of sum (k / r) v^T.  The token's own term, often far larger,
  // is added by one fma (as in the 64-token kernels).
  float acc[D], ks[D], own, vc, rinv;
#pragma unroll
  for (int j = 0; j < D; ++j) acc[j] = 0.f;
  const float* kb = a.k + b * a.T * Dr;
  const float* vb = a.v + b * a.T * M + cl;
  const float* rb = a.r + b * a.T;
  auto token = [&](int64_t s) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < D; ++j) ks[j] = ld_or_zero(kb + s * Dr, j, Dr);
    rinv = 1.0f / rb[s];
    const float kown = kb[s * Dr + rl], vown = vb[s * M];
    own = row_lane ? kown * rinv : 0.f;
    vc = col_lane ? vown : 0.f;
  };
  for (int64_t s0 = 0; s0 < t; s0 += 8) {
    float pa[D], px[D];
#pragma unroll
    for (int j = 0; j < D; ++j) pa[j] = px[j] = 0.f;
    const int64_t end = s0 + 8 < t ? s0 + 8 : t;
#pragma unroll 4
    for (int64_t s = s0; s < end; ++s) {
      token(s);
#pragma unroll
      for (int j = 0; j < D; ++j) {
        pa[j] = fmaf(own, ks[j], pa[j]);
        px[j] = fmaf(ks[j] * rinv, vc, px[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < D; ++j) {
      acc[j] += pa[j];
      x[j] += px[j];
    }
  }
  token(t);
#pragma unroll
  for (int j = 0; j < D; ++j) x[j] = fmaf(ks[j] * rinv, vc, x[j]);
  // L_t = inv(P0) + prefix, symmetrized through LDS, on the row owners.
  // Padded rows (lanes Dr .. D - 1) keep the identity.
  float lam[D];
#pragma unroll
  for (int j = 0; j < D; ++j) lam[j] = fmaf(own, ks[j], lam0[j] + acc[j]);
  if (lane < D) {
#pragma unroll
    for (int j = 0; j < D; ++j) tr[j * D + lane] = lam[j];
  }
  wave_fence();
  if (lane < D) {
#pragma unroll
    for (int j = 0; j < D; ++j) lam[j] = (lam[j] + tr[lane * D + j]) * 0.5f;
  }
  wave_fence();
  chol_rows<D>(lam, inv_diag, lane, mat, idg);  // mat = factor of L_t
  chol_solve<D>(mat, idg, x);
}

template <int D, bool EXACT>
__global__ __launch_bounds__(kWave) void scan_forward_short_kernel(ScanIn a, float* __restrict__ out,
                                                                   float* __restrict__ mT, float* __restrict__ cT) {
  __shared__ float mat[D * D], tr[D * D], idg[D];
  const int Dr = EXACT ? D : a.d, M = a.m, lane = threadIdx.x;
  const int64_t b = blockIdx.y, t = blockIdx.x;
  float x[D];
  token_state<D, EXACT>(a, b, t, lane, mat, tr, idg, x);
  const bool last = t == a.T - 1;
  if (lane < M) {
    const float* qt = a.q + (b * a.T + t) * Dr;
    float y = 0.f;
#pragma unroll
    for (int i = 0; i < D; ++i) y = fmaf(x[i], ld_or_zero(qt, i, Dr), y);
    out[(b * a.T + t) * M + lane] = y;
    if (last) {
#pragma unroll
      for (int i = 0; i < D; ++i)
        if (i < Dr) mT[(b * Dr + i) * M + lane] = x[i];
    }
  }
  if (last) {
    // P_T = L_T^{-1}: lane c solves for column c of the identity.
    float e[D];
#pragma unroll
    for (int i = 0; i < D; ++i) e[i] = lane == i ? 1.f : 0.f;
    chol_solve<D>(mat, idg, e);
    if (lane < Dr) {
#pragma unroll
      for (int i = 0; i < D; ++i)
        if (i < Dr) cT[(b * Dr + i) * Dr + lane] = e[i];
    }
  }
}

// The backward's passes (above) with a wave per token: gL_t [D, D] and gN_t [D,
// M], token by token in the workspace (in this order), their suffix sums in place
// (a thread an entry), then a wave per token again.  Sums as above: float64
// where gr would show their rounding.
template <int D, bool EXACT>
__global__ __launch_bounds__(kWave) void scan_backward_short_token_kernel(ScanIn a, const float* __restrict__ gy,
                                                                          const float* __restrict__ gmT,
                                                                          const float* __restrict__ gcT,
                                                                          float* __restrict__ ws_gl,
                                                                          float* __restrict__ ws_gn,
                                                                          float* __restrict__ gq) {
  __shared__ float mat[D * D], idg[D];
  __shared__ double tr[D * D];      // transpose staging
  __shared__ float mt[D * kMaxM];   // M_t, row-major
  __shared__ float gn[D * kMaxM];   // gN_t, row-major
  __shared__ float pt[D * D];       // P_T (last token); token_state's staging before it
  __shared__ float gys[kMaxM];
  const int Dr = EXACT ? D : a.d, M = a.m, lane = threadIdx.x;
  const int64_t b = blockIdx.y, t = blockIdx.x, row = b * a.T + t;
  const bool row_lane = lane < Dr, col_lane = lane < M, last = t == a.T - 1;
  float x[D];
  token_state<D, EXACT>(a, b, t, lane, mat, pt, idg, x);
  // Column owners: G[:, c] = q_t gy_t[c] (+ gM_T[:, c]), then gN[:, c] = L_t^{-1} G[:, c].
  float g[D];
  const float gyc = col_lane ? gy[row * M + lane] : 0.f;
#pragma unroll
  for (int i = 0; i < D; ++i) {
    float v = ld_or_zero(a.q + row * Dr, i, Dr) * gyc;
    if (last && gmT != nullptr && col_lane && i < Dr) v += gmT[(b * Dr + i) * M + lane];
    g[i] = col_lane ? v : 0.f;
  }
  chol_solve<D>(mat, idg, g);
  if (col_lane) {
    gys[lane] = gyc;
#pragma unroll
    for (int i = 0; i < D; ++i) {
      mt[i * kMaxM + lane] = x[i];
      gn[i * kMaxM + lane] = g[i];
      if (i < Dr) ws_gn[(row * Dr + i) * M + lane] = g[i];
    }
  }
  if (last && gcT != nullptr) {
    float e[D];
#pragma unroll
    for (int i = 0; i < D; ++i) e[i] = lane == i ? 1.f : 0.f;
    chol_solve<D>(mat, idg, e);  // lane c < D: column c of P_T (= row c)
    if (lane < D) {
#pragma unroll
      for (int i = 0; i < D; ++i) pt[lane * D + i] = e[i];
    }
  }
  wave_fence();
  // Row owners: gq_t[i] = sum_c M_t[i, c] gy_t[c] and row i of -gN_t M_t^T.
  double gl[D];
  if (lane < D) {
    double acc = 0.;
#pragma unroll
    for (int j = 0; j < D; ++j) gl[j] = 0.;
    for (int c = 0; c < M; ++c) {
      acc = fma(static_cast<double>(mt[lane * kMaxM + c]), static_cast<double>(gys[c]), acc);
      const double gc = -static_cast<double>(gn[lane * kMaxM + c]);
#pragma unroll
      for (int j = 0; j < D; ++j) gl[j] = fma(gc, static_cast<double>(mt[j * kMaxM + c]), gl[j]);
    }
    if (row_lane) gq[row * Dr + lane] = static_cast<float>(acc);
  }
  if (last && gcT != nullptr && lane < D) {
    // -(P_T gP_T P_T)[i][:]: row i of A = P_T gP_T in registers, then A P_T
    // (gP_T and the padded block of P_T: zero and the identity).
    float ar[D];
#pragma unroll
    for (int j = 0; j < D; ++j) {
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < D; ++k) {
        const float gkj = (k < Dr && j < Dr) ? gcT[(b * Dr + k) * Dr + j] : 0.f;
        acc = fmaf(pt[lane * D + k], gkj, acc);
      }
      ar[j] = acc;
    }
#pragma unroll
    for (int j = 0; j < D; ++j) {
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < D; ++k) acc = fmaf(ar[k], pt[k * D + j], acc);
      gl[j] -= acc;
    }
  }
  // Symmetrize through LDS and store row i of gL_t.
  if (lane < D) {
#pragma unroll
    for (int j = 0; j < D; ++j) tr[j * D + lane] = gl[j];
  }
  wave_fence();
  if (row_lane) {
#pragma unroll
    for (int j = 0; j < D; ++j)
      if (j < Dr) ws_gl[(row * Dr + lane) * Dr + j] = static_cast<float>((gl[j] + tr[lane * D + j]) * 0.5);
  }
}

// Loads run kSuffixBatch tokens ahead of the dependent sum.
constexpr int kSuffixBatch = 8;
__global__ __launch_bounds__(256) void scan_backward_short_suffix_kernel(float* __restrict__ ws_gl,
                                                                         float* __restrict__ ws_gn, int64_t T,
                                                                         int e_gl, int e_gn) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= e_gl + e_gn) return;
  const int64_t b = blockIdx.y;
  const bool gl = e < e_gl;
  const int w = gl ? e_gl : e_gn;
  float* p = gl ? ws_gl + b * T * e_gl + e : ws_gn + b * T * e_gn + (e - e_gl);
  double acc = 0.;
  int64_t t = T;
  while (t > 0) {
    const int n = t >= kSuffixBatch ? kSuffixBatch : static_cast<int>(t);
    float x[kSuffixBatch];
#pragma unroll
    for (int i = 0; i < kSuffixBatch; ++i) x[i] = i < n ? p[(t - 1 - i) * w] : 0.f;
#pragma unroll
    for (int i = 0; i < kSuffixBatch; ++i) {
      if (i < n) {
        acc += x[i];
        p[(t - 1 - i) * w] = static_cast<float>(acc);
      }
    }
    t -= n;
  }
}

template <int D, bool EXACT>
__global__ __launch_bounds__(kWave) void scan_backward_short_input_kernel(ScanIn a, const float* __restrict__ ws_gl,
                                                                          const float* __restrict__ ws_gn,
                                                                          float* __restrict__ gk,
                                                                          float* __restrict__ gv,
                                                                          float* __restrict__ gr,
                                                                          float* __restrict__ gm0,
                                                                          float* __restrict__ gc0) {
  __shared__ float mat[D * D], tmp[D * D], idg[D], sn[D * kMaxM];  // sn: SN_s, row-major
  __shared__ double part[kWave];
  const int Dr = EXACT ? D : a.d, M = a.m, lane = threadIdx.x;
  const int64_t b = blockIdx.y, s = blockIdx.x, row = b * a.T + s;
  const bool row_lane = lane < Dr, col_lane = lane < M;
  const int rl = row_lane ? lane : 0;
  // Suffix sums over t >= s: row owners row i of SL, column owners column c of SN.
  float sl[D], snc[D];
  const float* glt = ws_gl + (row * Dr + rl) * Dr;
  const float* gnt = ws_gn + row * Dr * M + (col_lane ? lane : 0);
#pragma unroll
  for (int j = 0; j < D; ++j) {
    const float l = glt[j < Dr ? j : 0], n = gnt[(j < Dr ? j : 0) * M];
    sl[j] = (row_lane && j < Dr) ? l : 0.f;
    snc[j] = (col_lane && j < Dr) ? n : 0.f;
  }
  if (col_lane) {
#pragma unroll
    for (int i = 0; i < D; ++i) sn[i * kMaxM + lane] = snc[i];
  }
  wave_fence();
  const float* ks = a.k + row * Dr;
  const float* vs = a.v + row * M;
  const float rinv = 1.0f / a.r[row];
  // gk_s[i] = (2 (SL k)_i + (SN v)_i) / r;  k^T SL k and k^T SN v for gr.
  double contrib = 0.;
  if (row_lane) {
    double l = 0., n = 0.;
#pragma unroll
    for (int j = 0; j < D; ++j) l = fma(static_cast<double>(sl[j]), static_cast<double>(ld_or_zero(ks, j, Dr)), l);
    for (int c = 0; c < M; ++c) n = fma(static_cast<double>(sn[lane * kMaxM + c]), static_cast<double>(vs[c]), n);
    gk[row * Dr + lane] = static_cast<float>(2. * l + n) * rinv;
    contrib = (l + n) * ks[lane];
  }
  part[lane] = contrib;
  if (col_lane) {
    double acc = 0.;
#pragma unroll
    for (int i = 0; i < D; ++i) acc = fma(static_cast<double>(snc[i]), static_cast<double>(ld_or_zero(ks, i, Dr)), acc);
    gv[row * M + lane] = static_cast<float>(acc) * rinv;
  }
  wave_fence();
  if (lane == 0) {
    double z = 0.;
    for (int i = 0; i < Dr; ++i) z += part[i];
    gr[row] = -static_cast<float>(z) * rinv * rinv;
  }
  if (s == 0) prior_grads<D>(a, b, Dr, lane, sl, snc, sn, mat, idg, tmp, gm0, gc0);
}

// Key dimensions 17..32: the general kernel with the matrices in LDS (a
// register-resident factor of that size would spill).  One wave per (b, t)
// as above; the factorization runs column by column in LDS.
// In-place Cholesky of the D x D matrix A (row-major in LDS); lower factor.
__device__ void lds_cholesky(float* A, int D, int lane) {
  for (int j = 0; j < D; ++j) {
    if (lane == 0) {
      float s = A[j * D + j];
      for (int k = 0; k < j; ++k) s = fmaf(-A[j * D + k], A[j * D + k], s);
      A[j * D + j] = sqrtf(s);
    }
    __syncthreads();
    const float piv = A[j * D + j];
    for (int i = j + 1 + lane; i < D; i += kWave) {
      float s = A[i * D + j];
      for (int k = 0; k < j; ++k) s = fmaf(-A[i * D + k], A[j * D + k], s);
      A[i * D + j] = s / piv;
    }
    __syncthreads();
  }
}

// Solve (L L^T) x = b for one right-hand side held by the calling lane.
__device__ void lds_chol_solve(const float* Lf, int D, float* x) {
  for (int i = 0; i < D; ++i) {
    float s = x[i];
    for (int k = 0; k < i; ++k) s = fmaf(-Lf[i * D + k], x[k], s);
    x[i] = s / Lf[i * D + i];
  }
  for (int i = D - 1; i >= 0; --i) {
    float s = x[i];
    for (int k = i + 1; k < D; ++k) s = fmaf(-Lf[k * D + i], x[k], s);
    x[i] = s / Lf[i * D + i];
  }
}

__global__ __launch_bounds__(kWave) void associative_scan_lds_kernel(const float* __restrict__ keys,
                                                                 const float* __restrict__ values,
                                                                 const float* __restrict__ queries,
                                                                 const float* __restrict__ obs,
                                                                 const float* __restrict__ mean0,
                                                                 const float* __restrict__ cov0,
                                                                 float* __restrict__ out, float* __restrict__ mT,
                                                                 float* __restrict__ cT, int64_t T, int D, int M) {
  __shared__ float C0[kMaxD * kMaxD];    // factor of P0
  __shared__ float Lam[kMaxD * kMaxD];   // precision, then its factor
  __shared__ float Nat[kMaxD * kMaxM];   // natural parameter
  __shared__ float Lam0[kMaxD * kMaxD];  // inv(P0)
  const int lane = threadIdx.x;
  const int64_t b = blockIdx.y;
  const int64_t t = blockIdx.x;
  const float* P0 = cov0 + b * D * D;
  const float* M0 = mean0 + b * D * M;

  // inv(P0) through its Cholesky factor (P0 is SPD).
  for (int e = lane; e < D * D; e += kWave) C0[e] = P0[e];
  __syncthreads();
  lds_cholesky(C0, D, lane);
  if (lane < D) {
    float x[kMaxD];
    for (int i = 0; i < D; ++i) x[i] = (i == lane) ? 1.f : 0.f;
    lds_chol_solve(C0, D, x);
    for (int i = 0; i < D; ++i) Lam0[i * D + lane] = x[i];
  }
  __syncthreads();

  // Prefix sums over s <= t, accumulated in token order.
  for (int e = lane; e < D * D; e += kWave) {
    const int i = e / D, j = e - i * D;
    float acc = 0.f;
    for (int64_t s = 0; s <= t; ++s) {
      const float* ks = keys + (b * T + s) * D;
      acc = fmaf(ks[i], ks[j] / obs[b * T + s], acc);
    }
    Lam[e] = Lam0[e] + acc;
  }
  for (int e = lane; e < D * M; e += kWave) {
    const int i = e / M, c = e - i * M;
    float acc = 0.f;
    for (int64_t s = 0; s <= t; ++s) {
      const float wk = keys[(b * T + s) * D + i] / obs[b * T + s];
      acc = fmaf(wk, values[(b * T + s) * M + c], acc);
    }
    float n0 = 0.f;
    for (int k = 0; k < D; ++k) n0 = fmaf(Lam0[i * D + k], M0[k * M + c], n0);
    Nat[e] = n0 + acc;
  }
  __syncthreads();
  // Symmetrise, then factor.
  for (int e = lane; e < D * D; e += kWave) {
    const int i = e / D, j = e - i * D;
    if (i < j) {
      const float v = (Lam[i * D + j] + Lam[j * D + i]) * 0.5f;
      Lam[i * D + j] = v;
      Lam[j * D + i] = v;
    }
  }
  __syncthreads();
  lds_cholesky(Lam, D, lane);

  const float* qt = queries + (b * T + t) * D;
  const bool last = (t == T - 1);
  for (int c = lane; c < M; c += kWave) {
    float x[kMaxD];
    for (int i = 0; i < D; ++i) x[i] = Nat[i * M + c];
    lds_chol_solve(Lam, D, x);
    float y = 0.f;
    for (int i = 0; i < D; ++i) y = fmaf(x[i], qt[i], y);
    out[(b * T + t) * M + c] = y;
    if (last)
      for (int i = 0; i < D; ++i) mT[b * D * M + i * M + c] = x[i];
  }
  if (last && lane < D) {
    float x[kMaxD];
    for (int i = 0; i < D; ++i) x[i] = (i == lane) ? 1.f : 0.f;
    lds_chol_solve(Lam, D, x);
    for (int i = 0; i < D; ++i) cT[b * D * D + i * D + lane] = x[i];
  }
}

// T == 0: the belief is the prior.
__global__ void copy_prior_kernel(const float* __restrict__ mean0, const float* __restrict__ cov0,
                                  float* __restrict__ mT, float* __restrict__ cT, int64_t nm, int64_t nc) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < nm) mT[i] = mean0[i];
  if (i < nc) cT[i] = cov0[i];
}

// Whether the kernels with a wave per token are the faster ones: fits of both
// sides' times at 24 pairs of batch (1 to 2048) and T (1 to 96) for each of 15
// key and value dimensions, at most 13 % off the faster side.  A workgroup of 64
// tokens takes the same time whatever T; it grows with the value columns, which
// its waves take in turn and a wave per token in lanes, as the latter grows with
// T.  While every token's wave has a SIMD of its own (1024; for twice as many the
// line is halved) the column solves decide: D = M = 16 forward, 16 x 16 tokens
// 16.9 against 22.3 us, 16 x 64 32.9 against 22.6; backward, 16 x 32 52.0 against
// 58.8, 16 x 64 69.1 against 59.5.  With more waves their work does: forward 2048
// x 4 59.5 against 103 us, 2048 x 8 132 against 103; backward 2048 x 8 322 against
// 484, 2048 x 16 668 against 496.  A key dimension that is padded costs the wave
// per token its branches.
bool short_sequences(bool backward, int64_t b, int64_t t, int d, int m) {
  const bool wide = d > 8, padded = d == 3 || (d > 4 && d != 8 && d != 16);
  int64_t idle, busy;
  if (backward) {
    idle = wide ? 22 + 2 * m : 4 + 7 * m / 10;
    if (padded) idle = idle * 3 / 5;
    busy = (wide ? 9 : 4) + m / 10;
  } else {
    idle = wide ? 12 + 6 * m / 5 : 1 + 7 * m / 10;
    if (padded) idle = idle * 7 / 20;
    busy = 4 + m / 8;
  }
  const int64_t waves = b * t;
  return t <= (waves <= 1024 ? idle : waves <= 2048 && idle / 2 > busy ? idle / 2 : busy);
}

template <int D, bool EXACT>
void launch_scan_backward_short(const ScanIn& a, const float* gy, const float* gmT, const float* gcT, float* ws,
                                float* gk, float* gv, float* gq, float* gr, float* gm0, float* gc0, int64_t b,
                                hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(a.T), static_cast<unsigned>(b)), block(kWave);
  float* ws_gl = ws;
  float* ws_gn = ws + b * a.T * a.d * a.d;
  hipLaunchKernelGGL((scan_backward_short_token_kernel<D, EXACT>), grid, block, 0, stream, a, gy, gmT, gcT, ws_gl,
                     ws_gn, gq);
  const int e_gl = a.d * a.d, e_gn = a.d * a.m;
  hipLaunchKernelGGL(scan_backward_short_suffix_kernel,
                     dim3(static_cast<unsigned>((e_gl + e_gn + 255) / 256), static_cast<unsigned>(b)), dim3(256), 0,
                     stream, ws_gl, ws_gn, a.T, e_gl, e_gn);
  hipLaunchKernelGGL((scan_backward_short_input_kernel<D, EXACT>), grid, block, 0, stream, a, ws_gl, ws_gn, gk, gv,
                     gr, gm0, gc0);
}

template <int D>
hipError_t launch_scan(const ScanIn& a, float* y, float* mT, float* cT, int64_t b, hipStream_t stream) {
  if (short_sequences(false, b, a.T, a.d, a.m)) {
    const dim3 grid(static_cast<unsigned>(a.T), static_cast<unsigned>(b)), block(kWave);
    if (a.d == D) hipLaunchKernelGGL((scan_forward_short_kernel<D, true>), grid, block, 0, stream, a, y, mT, cT);
    else hipLaunchKernelGGL((scan_forward_short_kernel<D, false>), grid, block, 0, stream, a, y, mT, cT);
    return hipGetLastError();
  }
  const dim3 grid(static_cast<unsigned>((a.T + kTok - 1) / kTok), static_cast<unsigned>(b)), block(kWaves * kWave);
  if (a.d == D && D % 4 == 0 && a.m % 4 == 0)
    hipLaunchKernelGGL((scan_forward_kernel<D, (D % 4 == 0)>), grid, block, 0, stream, a, y, mT, cT);
  else
    hipLaunchKernelGGL((scan_forward_kernel<D, false>), grid, block, 0, stream, a, y, mT, cT);
  return hipGetLastError();
}

template <int D, bool VEC>
void launch_scan_backward_vec(const ScanIn& a, const float* gy, const float* gmT, const float* gcT, const Ws& ws,
                              float* gk, float* gv, float* gq, float* gr, float* gm0, float* gc0, int64_t b,
                              hipStream_t stream) {
  const unsigned blocks = static_cast<unsigned>((a.T + kTok - 1) / kTok), rows = static_cast<unsigned>(b);
  const dim3 grid(blocks, rows), block(kWaves * kWave);
  hipLaunchKernelGGL((scan_backward_token_kernel<D, VEC>), grid, block, 0, stream, a, gy, gmT, gcT, ws, gq);
  const int entries = a.d * (a.d + 1) / 2 + a.d * a.m, per = kWaves * kPass2;
  hipLaunchKernelGGL(scan_backward_suffix_kernel, dim3(blocks, rows, static_cast<unsigned>((entries + per - 1) / per)),
                     block, 0, stream, ws, entries);
  hipLaunchKernelGGL((scan_backward_input_kernel<D, VEC>), grid, block, 0, stream, a, ws, gk, gv, gr, gm0, gc0);
}

template <int D>
hipError_t launch_scan_backward(const ScanIn& a, const float* gy, const float* gmT, const float* gcT, float* ws,
                                float* gk, float* gv, float* gq, float* gr, float* gm0, float* gc0, int64_t b,
                                hipStream_t stream) {
  if (short_sequences(true, b, a.T, a.d, a.m)) {
    if (a.d == D) launch_scan_backward_short<D, true>(a, gy, gmT, gcT, ws, gk, gv, gq, gr, gm0, gc0, b, stream);
    else launch_scan_backward_short<D, false>(a, gy, gmT, gcT, ws, gk, gv, gq, gr, gm0, gc0, b, stream);
    return hipGetLastError();
  }
  const Ws w{ws, a.T, a.d, a.m};
  if (a.d == D && D % 4 == 0 && a.m % 4 == 0)
    launch_scan_backward_vec<D, (D % 4 == 0)>(a, gy, gmT, gcT, w, gk, gv, gq, gr, gm0, gc0, b, stream);
  else
    launch_scan_backward_vec<D, false>(a, gy, gmT, gcT, w, gk, gv, gq, gr, gm0, gc0, b, stream);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_associative_scan_backward(const float* k, const float* v, const float* q, const float* r,
                                            const float* m0, const float* c0, const float* gy, const float* gmT,
                                            const float* gcT, float* ws, float* gk, float* gv, float* gq, float* gr,
                                            float* gm0, float* gc0, int64_t b, int64_t t, int d, int m,
                                            hipStream_t stream) {
  if (d > kMaxBackwardD || m > kMaxM || d <= 0 || m <= 0 || t <= 0 || t > 0x7fffffff || b > 65535)
    return hipErrorInvalidValue;
  if (b == 0) return hipSuccess;
  const ScanIn a{k, v, q, r, m0, c0, t, d, m};
  if (d <= 1) return launch_scan_backward<1>(a, gy, gmT, gcT, ws, gk, gv, gq, gr, gm0, gc0, b, stream);
  if (d <= 2) return launch_scan_backward<2>(a, gy, gmT, gcT, ws, gk, gv, gq, gr, gm0, gc0, b, stream);
  if (d <= 4) return launch_scan_backward<4>(a, gy, gmT, gcT, ws, gk, gv, gq, gr, gm0, gc0, b, stream);
  if (d <= 8) return launch_scan_backward<8>(a, gy, gmT, gcT, ws, gk, gv, gq, gr, gm0, gc0, b, stream);
  return launch_scan_backward<16>(a, gy, gmT, gcT, ws, gk, gv, gq, gr, gm0, gc0, b, stream);
}

hipError_t launch_associative_scan(const float* k, const float* v, const float* q, const float* r,
                                   const float* m0, const float* c0, float* y, float* mT, float* cT,
                                   int64_t b, int64_t t, int d, int m, hipStream_t stream) {
  if (d > kMaxD || m > kMaxM || d <= 0 || m <= 0) return hipErrorInvalidValue;
  if (b == 0) return hipSuccess;
  if (t == 0) {
    const int64_t nm = b * d * m, nc = b * d * d;
    const int64_t total = nm > nc ? nm : nc;
    hipLaunchKernelGGL(copy_prior_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, stream,
                       m0, c0, mT, cT, nm, nc);
    return hipGetLastError();
  }
  if (t > 0x7fffffff || b > 65535) return hipErrorInvalidValue;
  const ScanIn a{k, v, q, r, m0, c0, t, d, m};
  if (d <= 1) return launch_scan<1>(a, y, mT, cT, b, stream);
  if (d <= 2) return launch_scan<2>(a, y, mT, cT, b, stream);
  if (d <= 4) return launch_scan<4>(a, y, mT, cT, b, stream);
  if (d <= 8) return launch_scan<8>(a, y, mT, cT, b, stream);
  if (d <= 16) return launch_scan<16>(a, y, mT, cT, b, stream);
  hipLaunchKernelGGL(associative_scan_lds_kernel, dim3(static_cast<unsigned>(t), static_cast<unsigned>(b)),
                     dim3(kWave), 0, stream, k, v, q, r, m0, c0, y, mT, cT, t, d, m);
  return hipGetLastError();
}

}  // namespace bssm
