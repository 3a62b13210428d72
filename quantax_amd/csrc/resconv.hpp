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

constexpr int RC_WAVES = 4;
constexpr int RC_THREADS = RC_WAVES * WAVE;
constexpr int RC_MAXN = 1024;

// ---------------------------------------------------------------- layout
struct RcLayout {
  int nb, C, L0, L1, N, mode, actk;
  int win;                   // 16 x 16, C = 16: sliding-row-window forward and its K-step order
  int64_t nparams;
  int64_t off_l0w, off_l0b;  // first conv (Cin = 1): W (C, 9), b (C) in floats
  int64_t off_frag;          // start of per-layer fragment blocks (bytes)
  int64_t frag_bytes;        // bytes of one layer's fragments
  int64_t bias_off;          // start of per-layer biases (floats, (2nb) x C)
  int64_t off_jac;           // start of the Jacobian's FP32 fragments (bytes), see rc_pack_jac_kernel
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

template <int C, int MODE>
struct RcK {
  static constexpr int CT = C / 16;                                   // output-channel tiles
  static constexpr int KS = (MODE == QTX_CONV_FP32) ? (9 * C / 4) : (C == 16 ? 5 : 9);  // K steps
  static constexpr int CH = C / 4;                                    // 16-byte chunks per position
  static constexpr int FRAG_WORDS = (MODE == QTX_CONV_FP32) ? 1 : 8;  // 4-byte words per lane per (ct, ks)
};

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
  int ct = L.C / 16;
  int ks = (L.mode == QTX_CONV_FP32) ? 9 * L.C / 4 : (L.C == 16 ? (L.win ? 6 : 5) : 9);
  int words = (L.mode == QTX_CONV_FP32) ? 1 : 8;
  L.frag_bytes = (int64_t)ct * ks * WAVE * words * 4;
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
