// What the ResConv kernels share: the packed-parameter layout, the lattice
// geometry, the activations and the argument checks.
#pragma once
#include <cmath>
#include <string>

#include "common.hpp"

namespace qtx {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int RC_MAXN = 1024;

// ---------------------------------------------------------------- layout
struct RcLayout {
  int nb, C, L0, L1, N, mode, actk;
  int win;                   // 16 x 16, C = 16: sliding-row-window forward and its K-step order
  int64_t nparams;
  int64_t off_l0w, off_l0b;  // first conv (Cin = 1): W (C, 9), b (C) in floats
  int64_t off_frag;          // start of per-layer fragment blocks (bytes)
  int64_t frag_bytes;        // bytes of one layer's fragments, see rc_frag_steps
  int64_t bias_off;          // start of per-layer biases (floats, (2nb) x C)
  int64_t off_jac;           // start of the Jacobian's FP32 fragments (bytes), see rc_pack_kernel
  int64_t total_bytes;
};

__host__ __device__ inline int64_t rc_nparams(int nb, int C) {
  int64_t n = 0;
  for (int i = 0; i < nb; ++i) {
    int cin = (i == 0) ? 1 : C;
    n += (int64_t)C * cin * 9 + C;                 // conv1 (+ bias)
    n += (int64_t)C * C * 9 + ((i == nb - 1) ? 0 : C);  // conv2 (+ bias except last)
  }
  return n;
}

// offsets of layer l's weight/bias in the ravel_pytree vector
__host__ __device__ inline void rc_theta_offsets(int nb, int C, int l, int64_t& w, int64_t& b) {
  int64_t off = 0;
  for (int ll = 0; ll < 2 * nb; ++ll) {
    int i = ll / 2;
    int cin = (ll == 0) ? 1 : C;
    bool hb = !((ll % 2 == 1) && (i == nb - 1));
    if (ll == l) {
      w = off;
      b = hb ? off + (int64_t)C * cin * 9 : -1;
      return;
    }
    off += (int64_t)C * cin * 9 + (hb ? C : 0);
  }
  w = b = -1;
}

// 64-lane fragments of one layer at off_frag: none for the any-lattice FP32 kernels,
// which read the Jacobian's
inline int64_t rc_frag_steps(const RcLayout& L) {
  const int ct = L.C / 16;
  if (L.mode == QTX_CONV_FP32) return L.win ? ct * 9 * L.C / 4 : 0;
  return ct * (L.C == 16 ? (L.win ? 6 : 5) : 9);
}

inline RcLayout rc_layout(const qtx_resconv_desc* d) {
  RcLayout L;
  L.nb = d->nblocks;
  L.C = d->channels;
  L.L0 = d->L0;
  L.L1 = d->L1;
  L.N = d->L0 * d->L1;
  L.mode = d->precision;
  L.actk = d->activation;
  L.win = (L.C == 16 && L.L0 == 16 && L.L1 == 16) ? 1 : 0;
  L.nparams = rc_nparams(L.nb, L.C);
  int64_t off = L.nparams * 4;  // raw theta copy first
  off = (off + 255) & ~(int64_t)255;
  L.off_l0w = off / 4;
  off += (int64_t)L.C * 9 * 4;
  L.off_l0b = off / 4;
  off += (int64_t)L.C * 4;
  off = (off + 255) & ~(int64_t)255;
  L.bias_off = off / 4;
  off += (int64_t)2 * L.nb * L.C * 4;
  off = (off + 255) & ~(int64_t)255;
  L.off_frag = off;
  L.frag_bytes = rc_frag_steps(L) * WAVE * (L.mode == QTX_CONV_FP32 ? 1 : 8) * 4;
  off += L.frag_bytes * 2 * L.nb;  // slot per layer index (slot 0 unused)
  off = (off + 255) & ~(int64_t)255;
  L.off_jac = off;
  off += (int64_t)2 * L.nb * 2 * L.C * L.C * 9 * 4;
  L.total_bytes = off;
  return L;
}

// ---------------------------------------------------------------- math
// Activations (qtx_resconv_desc.activation): QTX_ACT_GELU_TANH, the
// reference's jax.nn.gelu default (model/conv_nets.py:85, 87),
// QTX_ACT_GELU_ERF, and QTX_ACT_RELU (max(x, 0), derivative 0 at x <= 0, as
// jax.nn.relu), an opt-in variant with no counterpart in the reference.
// tanh form: 0.5 x (1 + tanh(k (x + 0.044715 x^3))) = x / (1 + 2^(x (A + B x^2)))
// with A = -2 k log2(e), B = -2 k 0.044715 log2(e), k = sqrt(2 / pi); native exp2 and rcp
__device__ __forceinline__ float act_f(float x, int actk) {
  if (actk == QTX_ACT_RELU) return fmaxf(x, 0.0f);
  if (actk == QTX_ACT_GELU_ERF) return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f));
  constexpr float A = -2.0f * 0.79788456080286536f * 1.4426950408889634f;
  constexpr float Bc = A * 0.044715f;
  float e = __builtin_amdgcn_exp2f(x * fmaf(x * x, Bc, A));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

__device__ __forceinline__ float act_grad_f(float x, int actk) {
  if (actk == QTX_ACT_RELU) return x > 0.0f ? 1.0f : 0.0f;
  if (actk == QTX_ACT_GELU_ERF)
    return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * __expf(-0.5f * x * x) * 0.39894228040143268f;
  float u = 0.79788456080286536f * (x + 0.044715f * x * x * x);
  float t = 1.0f - 2.0f / (1.0f + __expf(2.0f * u));
  return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * 0.79788456080286536f * (1.0f + 0.134145f * x * x);
}

struct RcGeom {
  int L0, L1, N, NT;
  double log_cn;  // log(C N): the head's normalisation
};

__device__ __forceinline__ int tap_pos(const RcGeom& g, int y, int x, int tap) {
  int dy = tap / 3 - 1, dx = tap % 3 - 1;
  int ys = y + dy, xs = x + dx;
  ys = ys < 0 ? ys + g.L0 : (ys >= g.L0 ? ys - g.L0 : ys);
  xs = xs < 0 ? xs + g.L1 : (xs >= g.L1 ? xs - g.L1 : xs);
  return ys * g.L1 + xs;
}

// act(sc x) and act'(sc x) of four values, one branch on the activation
__device__ __forceinline__ v4f act4(v4f x, float sc, int actk) {
  v4f o;
  if (actk == QTX_ACT_GELU_TANH) {
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = act_f(x[q] * sc, QTX_ACT_GELU_TANH);
  } else if (actk == QTX_ACT_RELU) {
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = act_f(x[q] * sc, QTX_ACT_RELU);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = act_f(x[q] * sc, QTX_ACT_GELU_ERF);
  }
  return o;
}

__device__ __forceinline__ v4f act_grad4(v4f x, float sc, int actk) {
  v4f o;
  if (actk == QTX_ACT_GELU_TANH) {
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = act_grad_f(x[q] * sc, QTX_ACT_GELU_TANH);
  } else if (actk == QTX_ACT_RELU) {
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = act_grad_f(x[q] * sc, QTX_ACT_RELU);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = act_grad_f(x[q] * sc, QTX_ACT_GELU_ERF);
  }
  return o;
}

// v = hi + lo + O(2^-16 |v|): hi = bf16(v) (round to nearest even), lo =
// bf16(v - hi).  v - hi is formed by v_dot2c_f32_bf16 from the packed hi
// pair, (hi0, hi1) . (-1, 0) + v0 and (hi0, hi1) . (0, -1) + v1, exact
// (bf16 products are exact in FP32 and v - hi is representable), so hi is
// never widened back to FP32 by bit moves.
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split_bf16x4(v4f v, v4bf& hi, v4bf& lo) {
  const v2bf h01 = {(__bf16)v[0], (__bf16)v[1]}, h23 = {(__bf16)v[2], (__bf16)v[3]};
  // the selectors come from registers: an inline constant here (the
  // compiler encodes e0 as "-1.0") is not read as (bf16 -1, 0) by the hardware
  uint32_t u0 = 0x0000bf80u, u1 = 0xbf800000u;
  asm("" : "+v"(u0), "+v"(u1));
  const v2bf e0 = __builtin_bit_cast(v2bf, u0), e1 = __builtin_bit_cast(v2bf, u1);
  const float l0 = __builtin_amdgcn_fdot2_f32_bf16(h01, e0, v[0], false);
  const float l1 = __builtin_amdgcn_fdot2_f32_bf16(h01, e1, v[1], false);
  const float l2 = __builtin_amdgcn_fdot2_f32_bf16(h23, e0, v[2], false);
  const float l3 = __builtin_amdgcn_fdot2_f32_bf16(h23, e1, v[3], false);
  const v2bf l01 = {(__bf16)l0, (__bf16)l1}, l23 = {(__bf16)l2, (__bf16)l3};
  hi = v4bf{h01[0], h01[1], h23[0], h23[1]};
  lo = v4bf{l01[0], l01[1], l23[0], l23[1]};
}

struct RcArgs {
  RcGeom g;
  int nb, actk;
  const char* packed;
  int64_t off_l0w, off_l0b, bias_off, off_frag, frag_bytes, off_jac;
};

// Wait out the MFMAs that wrote acc[0 .. N) before any use of them.  The
// compiler counts the wait states behind an MFMA along the fall-through path
// only: a use reached over a short branch can read a result (or overwrite a
// register) too early.  Volatile asm statements keep their order: the first
// pass puts every MFMA before the wait, the second every use after it.
template <int N>
__device__ __forceinline__ void mfma_settle(v4f* acc) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(acc[i]));
  asm volatile("s_nop 15" : "+v"(acc[0]));
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(acc[i]));
}

// psi(s') / psi(s) = e^d for the local energy: 2^t, t = d log2(e), split
// into an integer k applied exactly by ldexp and f = t - k in [-1/2, 1/2]
// whose 2^f is one FP32 exp2 (about 1 ulp); the FP64 product d log2(e) and
// the FP32 rounding of f keep the relative error near 1e-7 for any d, where
// an FP32 exp of d itself would lose |d| * 2^-24 to the rounding of d alone.
// |t| >= 2100 is exp's overflow (+inf) or underflow (0) outright, and NaN
// stays NaN: no FP64 exp, whose polynomial constants would otherwise occupy
// VGPRs for the whole kernel.
__device__ __forceinline__ double exp_ratio(double d) {
  const double t = d * 1.4426950408889634;
  if (!(fabs(t) < 2100.0)) return d > 0.0 ? HUGE_VAL : (d < 0.0 ? 0.0 : d);  // exp's overflow / underflow; NaN stays
  const double k = rint(t);
  return ldexp((double)__builtin_amdgcn_exp2f((float)(t - k)), (int)k);
}

static inline int rc_check(const qtx_resconv_desc* d) {
  QTX_REQUIRE(d != nullptr, "null qtx_resconv_desc");
  QTX_REQUIRE(d->channels == 16 || d->channels == 32, "channels must be 16 or 32");
  QTX_REQUIRE(d->nblocks >= 1 && d->nblocks <= 64, "nblocks out of range (1..64)");
  QTX_REQUIRE(d->L0 >= 1 && d->L1 >= 1 && d->L0 * d->L1 <= RC_MAXN, "L0 * L1 out of range (1..1024)");
  QTX_REQUIRE(d->precision == QTX_CONV_FP32 || d->precision == QTX_CONV_BF16X3, "unknown precision");
  QTX_REQUIRE(d->activation == QTX_ACT_GELU_TANH || d->activation == QTX_ACT_GELU_ERF ||
                  d->activation == QTX_ACT_RELU,
              "unknown activation");
  if (d->channels == 16) QTX_REQUIRE(d->L0 * d->L1 <= 512, "channels = 16 needs L0 * L1 <= 512");
  if (d->channels == 32) QTX_REQUIRE(d->L0 * d->L1 <= 400, "channels = 32 needs L0 * L1 <= 400");
  return QTX_OK;
}

}  // namespace qtx
