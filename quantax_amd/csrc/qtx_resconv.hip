// ResConv(nblocks, C, 3) on a periodic L0 x L1 grid: batched forward on MFMA
// (FP32 16x16x4, or split-bf16 16x16x32 with FP32 accumulation), Metropolis
// with one full forward per proposal and local energy over connected
// configurations generated in LDS.
//
// The 16 x 16 window kernels and the large 32-channel split-bf16 ones are here,
// every other shape in resconv_wave.hpp.  The residual stream stays in
// registers in the MFMA output layout (lane l: channel 16 ct + 4 (l / 16) + q,
// site 16 t + l % 16).
//
// LDS activations: per configuration, per site, C/4 chunks of 16 bytes,
// XOR-swizzled so the eight lanes a ds_read_b128 serves at a time (eight
// consecutive sites) hit distinct 16-byte bank groups.
//   FP32   : chunk j = channels 4j .. 4j+3 (float)
//   BF16X3 : chunk j < C/8 = hi(channels 8j .. 8j+7), chunk C/8 + j = lo(...)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>

#include "resconv_wave.hpp"

namespace qtx {

// ---------------------------------------------------------------- packing
// one thread per (layer, ct, ks, lane) fragment for layers 1 .. 2nb-1
template <int C, int MODE, int WIN>
__global__ void rc_pack_frag_kernel(const float* __restrict__ theta, int nb, char* __restrict__ packed,
                                    int64_t off_frag, int64_t frag_bytes) {
  constexpr int KCT = C / 16;
  constexpr int KKS = (MODE == QTX_CONV_FP32) ? 9 * C / 4 : (C == 16 ? (WIN ? 6 : 5) : 9);
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t per_layer = (int64_t)KCT * KKS * WAVE;
  int64_t total = per_layer * (2 * nb - 1);
  if (idx >= total) return;
  int l = 1 + (int)(idx / per_layer);
  int64_t rem = idx % per_layer;
  int ct = (int)(rem / (KKS * WAVE));
  int ks = (int)((rem / WAVE) % KKS);
  int lane = (int)(rem % WAVE);
  int64_t w0, b0;
  rc_theta_offsets(nb, C, l, w0, b0);
  const int co = 16 * ct + lane % 16, g = lane / 16;
  // window layout, split-bf16: conv1 layers l >= 2 carry the scale of the
  // conv2 before them, which then outputs act(s x) / s
  const float wsc = (WIN && MODE == QTX_CONV_BF16X3 && l >= 2 && (l % 2) == 0) ? 1.0f / sqrtf((float)(l / 2 + 1)) : 1.0f;
  auto W = [&](int ci, int tap) -> float { return theta[w0 + ((int64_t)co * C + ci) * 9 + tap] * wsc; };
  char* dst = packed + off_frag + (int64_t)l * frag_bytes;
  if constexpr (MODE == QTX_CONV_FP32) {
    // ks = (tap, h, j'): ci = 16 h + 4 g + j'
    int tap = ks / (C / 4), rr = ks % (C / 4), h = rr / 4, jp = rr % 4;
    float v = W(16 * h + 4 * g + jp, tap);
    reinterpret_cast<float*>(dst)[((int64_t)ct * KKS + ks) * WAVE + lane] = v;
  } else {
    int tap, c0;
    // window layout: per K-step a plane of 64 x 16 B slot-0 fragments, then
    // one of slot-1 fragments (16-byte lane stride for the LDS reads);
    // other layouts: the two slots of a lane side by side
    __bf16* o = reinterpret_cast<__bf16*>(dst) + (((int64_t)ct * KKS + ks) * WAVE + lane) * 16;
    __bf16* o1 = o + 8;
    if (WIN) {
      o = reinterpret_cast<__bf16*>(dst) + ((((int64_t)ct * KKS + ks) * 2) * WAVE + lane) * 8;
      o1 = o + WAVE * 8;
    }
    if (WIN && (ks % 2) == 1) {
      // tap (dy, 2) holds 16 of a K-step's 32 rows, so its three split
      // products share instructions: slot 0 of K-step 2 dy + 1 is
      // [hi | lo] of tap (dy, 2) (against [X hi; X hi]); slot 1 carries the
      // hi-times-X-lo halves: [hi (0, 2) | hi (1, 2)] in K-step 1,
      // [hi (2, 2) | 0] in K-step 3, zeros in K-step 5
      const int dy = ks / 2, up = g >> 1;
      c0 = 8 * (g & 1);
      for (int q = 0; q < 8; ++q) {
        const float v = W(c0 + q, 3 * dy + 2);
        const __bf16 hi = (__bf16)v;
        o[q] = up ? (__bf16)(v - (float)hi) : hi;
        float v1 = 0.0f;
        if (dy == 0) v1 = W(c0 + q, up ? 5 : 2);
        else if (dy == 1 && !up) v1 = W(c0 + q, 8);
        o1[q] = (__bf16)v1;
      }
      return;
    }
    if (WIN) {
      // ks = 2 dy: taps (dy, 0), (dy, 1)
      tap = 3 * (ks / 2) + (g >> 1);
      c0 = 8 * (g & 1);
    } else if (C == 16) {
      tap = 2 * ks + (g >> 1);
      c0 = 8 * (g & 1);
    } else {
      tap = ks;
      c0 = 8 * g;
    }
    for (int q = 0; q < 8; ++q) {
      float v = (tap < 9) ? W(c0 + q, tap) : 0.0f;
      __bf16 hi = (__bf16)v;
      __bf16 lo = (__bf16)(v - (float)hi);
      o[q] = hi;
      o1[q] = lo;
    }
  }
}

// Everything but the fragments of rc_pack_frag_kernel, in one launch: the copy of
// theta, layer 0's weights and bias, the layers' biases, and the FP32 A fragments
// of layers 1 .. 2nb-1, which the Jacobian reads whatever the forward's precision and
// the any-lattice FP32 forward reads too: per layer and direction (0: forward, 1:
// input gradient, with the two channel indices exchanged and the taps mirrored)
// [tap][row tile][column half][lane][4]: row = 16 ct + lane % 16, column = 16 h +
// 4 (lane / 16) + j, so a lane reads its four K values of a tap in one 16-byte load
template <int C>
__global__ void rc_pack_kernel(const float* __restrict__ theta, int nb, int64_t nparams, float* __restrict__ packed,
                               int64_t off_l0w, int64_t off_l0b, int64_t bias_off, float* __restrict__ frag) {
  constexpr int CT = C / 16;
  constexpr int64_t per = (int64_t)C * C * 9;
  int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < nparams) {
    packed[j] = theta[j];
    return;
  }
  j -= nparams;
  if (j < C * 9) {
    packed[off_l0w + j] = theta[j];  // layer 0 weights start at 0
    return;
  }
  j -= C * 9;
  if (j < C) {
    packed[off_l0b + j] = theta[C * 9 + j];
    return;
  }
  j -= C;
  if (j < (int64_t)2 * nb * C) {
    const int l = (int)(j / C), co = (int)(j % C);
    int64_t w0, b0;
    rc_theta_offsets(nb, C, l, w0, b0);
    packed[bias_off + j] = (b0 >= 0) ? theta[b0 + co] : 0.0f;
    return;
  }
  j -= (int64_t)2 * nb * C;
  if (j >= (int64_t)(2 * nb - 1) * 2 * per) return;
  const int l = 1 + (int)(j / (2 * per)), dir = (int)(j / per) & 1;
  const int e = (int)(j % per);
  const int i = e % 4, lane = (e / 4) % WAVE, h = (e / 256) % CT, ct = (e / 256 / CT) % CT, tap = e / 256 / CT / CT;
  const int row = 16 * ct + lane % 16, col = 16 * h + 4 * (lane / 16) + i;
  const int64_t w0 = 10 * C + (int64_t)(l - 1) * (per + C);  // layer l >= 1 of rc_theta_offsets
  frag[((int64_t)l * 2 + dir) * per + e] =
      dir == 0 ? theta[w0 + ((int64_t)row * C + col) * 9 + tap] : theta[w0 + ((int64_t)col * C + row) * 9 + (8 - tap)];
}

// ---------------------------------------------------------------- forwards
// Sliding-row-window forward for C = 16 on a 16 x 16 grid.  Workgroup:
// WPC B waves, B configurations; wave w owns the RPW = 16 / WPC rows
// RPW (w % WPC) .. of configuration w / WPC and walks them in order keeping
// the B fragments of input rows y - 1, y, y + 1 in registers: every fragment
// depends only on its input row (split-bf16 K-steps 2 dy + pr: pr 0 = taps
// (dy, 0) + (dy, 1), pr 1 = tap (dy, 2) in both K halves, whose split
// products over the three dy take five instructions per output row, see the
// packing; FP32 K-steps = taps), so each row is read from LDS once per wave
// and layer instead of three times.  The hi-times-X-lo halves of tap (dy, 2)
// pair rows y - 1 and y in one instruction: the lo fragment of row r is
// loaded with its upper K half (lanes 32-63) from row r + 1, so
// [X lo (y - 1); X lo (y)] is row y - 1's fragment as loaded, with no lane
// select per row.  With split-bf16, a conv1 layer's packed weights carry the
// scale s of the conv2 before it, whose epilogue then writes act(s x) / s
// (s folds into the activation's constants: one multiply per value less).
//
// Issue structure: the activation and the conv kind (conv1 / conv2 with
// residual) are compile-time inside a layer (one branch per layer), and the
// rows are software-pipelined: row i's MFMA chain and row i - 1's epilogue
// (residual, activation, bf16 split, LDS store) are one basic block, so VALU
// and MFMA work of the same wave can overlap.  Every wave reads layer l's
// weight fragments from one LDS stage (wst, RC_WSTAGE bytes) into registers
// at the layer start, together with its first two input rows and the row
// after its last (the latter two belong to the configuration's other waves);
// after a barrier, layer l + 1's fragments travel HBM/L2 -> LDS by DMA into
// the same stage while layer l runs, and each wave writes its output rows in
// place of its input rows (one activation buffer per configuration).  The
// residual stream x (FP32, 4 values per lane and row) stays in registers.
// Dispatched with WPC = 2, B = 2 (8 rows per wave, 46-52 KB of LDS and at
// most 256 VGPRs, two workgroups per CU): against WPC = 4, B = 1 (4 rows,
// ping-pong buffers, three workgroups per CU at 168 VGPRs) the per-layer
// prologue and pipeline drain are spread over twice the rows, and E_loc at
// 16 x 16 runs at 290 against 283 TFLOP/s (352 against 334 with ReLU).
constexpr int RC_WSTAGE = 12288;  // one layer's fragments: bf16x3 6 x 64 x 32 B; FP32 9216 B
constexpr int RC_WBIAS = 64;     // the layer's 16 FP32 biases, after the fragments
constexpr int rc_win_lds(int B) { return RC_WSTAGE + RC_WBIAS; }  // one weight stage
typedef __attribute__((address_space(3))) void rc_lds_void;

template <int ACT>
__device__ __forceinline__ float act_t(float x) {
  return act_f(x, ACT);
}

// act(s x) / s for s > 0, with the layer constants k0 = s A, k1 = s^3 B (tanh
// GELU) or k0 = s / sqrt(2) (erf GELU)
template <int ACT>
__device__ __forceinline__ float act_over_s(float x, float k0, float k1) {
  if constexpr (ACT == QTX_ACT_RELU) return fmaxf(x, 0.0f);
  else if constexpr (ACT == QTX_ACT_GELU_ERF) return 0.5f * x * (1.0f + erff(x * k0));
  else return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * fmaf(x * x, k1, k0)));
}

template <int MODE, int B, int WPC>
__device__ __attribute__((always_inline)) inline void rc_forward_win(
    const RcGeom& g, int nb, int actk, const char* __restrict__ packed, int64_t off_l0w, int64_t off_l0b,
    int64_t bias_off, int64_t off_frag, int64_t frag_bytes, const int8_t* sp, char* act, char* wst, float* red,
    double* lp_out) {
  constexpr int C = 16, W = WPC * B, L0 = 16, RPW = L0 / WPC;
  constexpr int ROWB = 16 * 64;
  constexpr int CFGB = L0 * ROWB;
  constexpr int KSW = (MODE == QTX_CONV_FP32) ? 36 : 6;
  // the lane index through an opaque move: every per-lane address below is
  // then computed inside the forward instead of being hoisted into
  // registers held (or spilled) across a caller's whole loop
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid % WAVE, wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int gq = lane / 16, x = lane % 16;
  const int b = wv / WPC, y0 = RPW * (wv % WPC);
  const float* pf = reinterpret_cast<const float*>(packed);

  // the 16-byte chunks of column c (64 bytes per column) are XORed with
  // (c >> 1) & 3: the eight lanes a ds_read_b128 serves per cycle read eight
  // consecutive columns, which then fall on distinct 16-byte bank groups
  // (with (c >> 2) & 3 columns c and c + 2 collide: the sweep is 6.6 % slower)
  int xoff[3];
#pragma unroll
  for (int dx = 0; dx < 3; ++dx) {
    int xs = (x + dx + 15) & 15;
    xoff[dx] = xs * 64 + ((gq ^ ((xs >> 1) & 3)) << 4);
  }
  int khi[2], klo[2];
#pragma unroll
  for (int pr = 0; pr < 2; ++pr) {
    int dx = (pr == 0) ? (gq >> 1) : 2;
    int xs = (x + dx + 15) & 15, key = (xs >> 1) & 3, jh = gq & 1;
    khi[pr] = xs * 64 + ((jh ^ key) << 4);
    klo[pr] = xs * 64 + (((2 + jh) ^ key) << 4);
  }
  const int key0 = (x >> 1) & 3;
  const int st_f32 = x * 64 + ((gq ^ key0) << 4);
  const int st_hi = x * 64 + (((gq >> 1) ^ key0) << 4) + (gq & 1) * 8;
  const int st_lo = x * 64 + (((2 + (gq >> 1)) ^ key0) << 4) + (gq & 1) * 8;
  auto store4 = [&](char* row_base, v4f v) {
    if constexpr (MODE == QTX_CONV_FP32) {
      *reinterpret_cast<v4f*>(row_base + st_f32) = v;
    } else {
      v4bf hi, lo;
      split_bf16x4(v, hi, lo);
      *reinterpret_cast<v4bf*>(row_base + st_hi) = hi;
      *reinterpret_cast<v4bf*>(row_base + st_lo) = lo;
    }
  };

  // B fragments of one input row
  struct Frag {
    v4f f[(MODE == QTX_CONV_FP32) ? 3 : 1];
    v8bf h[(MODE == QTX_CONV_FP32) ? 1 : 2];
    v8bf l[(MODE == QTX_CONV_FP32) ? 1 : 2];
  };
  const int klo1n = klo[1] + (lane >= 32 ? ROWB : 0);
  // nxt: the upper K half of F.l[1] comes from row r + 1 (no wrap), else row r
  auto load_row = [&](const char* cfg, int r, bool nxt) {
    Frag F;
    const char* rb = cfg + ((r + L0) & (L0 - 1)) * ROWB;
    if constexpr (MODE == QTX_CONV_FP32) {
#pragma unroll
      for (int dx = 0; dx < 3; ++dx) F.f[dx] = *reinterpret_cast<const v4f*>(rb + xoff[dx]);
    } else {
#pragma unroll
      for (int pr = 0; pr < 2; ++pr) F.h[pr] = *reinterpret_cast<const v8bf*>(rb + khi[pr]);
      F.l[0] = *reinterpret_cast<const v8bf*>(rb + klo[0]);
      F.l[1] = *reinterpret_cast<const v8bf*>(rb + (nxt ? klo1n : klo[1]));
    }
    return F;
  };
  // layer l's fragment block -> the weight stage, frag_bytes / 1024 wave-wide DMA instructions
  auto stage_weights = [&](int l) {
    const char* src = packed + off_frag + (int64_t)l * frag_bytes;
    char* dst = wst;
    const int nchunk = (int)(frag_bytes >> 10);
    for (int c = wv; c < nchunk; c += W)
      __builtin_amdgcn_global_load_lds((const void*)(src + c * 1024 + lane * 16), (rc_lds_void*)(dst + c * 1024), 16,
                                       0, 0);
    // the biases travel with the fragments: read from global memory at the
    // layer start, the first MFMA would wait for the whole DMA as well
    if (wv == W - 1 && lane < C / 4)
      __builtin_amdgcn_global_load_lds((const void*)(packed + bias_off * 4 + (int64_t)l * C * 4 + lane * 16),
                                       (rc_lds_void*)(dst + RC_WSTAGE), 16, 0, 0);
  };

  v4f resr[RPW];  // residual stream of the wave's rows, MFMA output layout
  stage_weights(1);
  // ---- layer 0 on VALU
  {
    // this lane's 4 output channels 4 gq + q: weights from one base
    const float* W0 = pf + off_l0w + 4 * gq * 9;
    const float* b0 = pf + off_l0b + 4 * gq;
    // an opaque zero keeps the 9 x RPW spin addresses from being hoisted out
    // of the forward (they would be held, or spilled, for the whole kernel)
    int z0 = 0;
    asm volatile("" : "+s"(z0));
    const int8_t* s = sp + b * 256 + z0;
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const int y = y0 + i;
      float sv[9];
#pragma unroll
      for (int tap = 0; tap < 9; ++tap)
        sv[tap] = (float)s[((y + tap / 3 - 1 + L0) & (L0 - 1)) * 16 + ((x + tap % 3 + 15) & 15)] *
                  0.70710678118654752f;
      float spin = (float)s[y * 16 + x];
      v4f z;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float a = b0[q];
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) a += W0[q * 9 + tap] * sv[tap];
        z[q] = act_f(a, actk);
      }
      resr[i] = v4f{spin, spin, spin, spin};
      store4(act + b * CFGB + y * ROWB, z);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's weight DMA has landed
  __syncthreads();

  // one layer: weights from the LDS stage, rows software-pipelined; EPI is
  // called with (row, accumulator)
  auto run_layer = [&](int l, const char* in, auto&& epi) {
    // rows y0 - 1 and y0 + RPW belong to the configuration's other waves:
    // read before the barrier below, after which every wave overwrites its
    // own rows in place
    Frag Fm = load_row(in, y0 - 1, false);
    if constexpr (MODE != QTX_CONV_FP32) {
      // [X lo (y0 - 1); X lo (y0)]: row y0 - 1 may wrap
      const char* pm = (lane < 32) ? in + ((y0 - 1 + L0) & (L0 - 1)) * ROWB : in + y0 * ROWB;
      Fm.l[1] = *reinterpret_cast<const v8bf*>(pm + klo[1]);
    }
    Frag F0 = load_row(in, y0, true);
    Frag Fe = load_row(in, y0 + RPW, false);
    float wf[(MODE == QTX_CONV_FP32) ? KSW : 1];
    v8bf wh[(MODE == QTX_CONV_FP32) ? 1 : KSW];
    v8bf wl[(MODE == QTX_CONV_FP32) ? 1 : KSW];
    const char* fr = wst;
    if constexpr (MODE == QTX_CONV_FP32) {
#pragma unroll
      for (int i = 0; i < KSW; ++i) wf[i] = reinterpret_cast<const float*>(fr)[i * WAVE + lane];
    } else {
#pragma unroll
      for (int i = 0; i < KSW; ++i) {
        const v8bf* src = reinterpret_cast<const v8bf*>(fr) + 2 * i * WAVE + lane;
        wh[i] = src[0];
        wl[i] = src[WAVE];
      }
    }
    const v4f bias4 = *reinterpret_cast<const v4f*>(fr + RC_WSTAGE + 16 * gq);
    // every wave holds this layer's fragments: the next layer's travel into
    // the stage while this one runs
    __syncthreads();
    if (l + 1 < 2 * nb) stage_weights(l + 1);
    v4f accp = bias4;
#pragma unroll
    for (int i = 0; i <= RPW; ++i) {
      v4f acc = bias4;
      Frag Fp;
      if (i < RPW) {
        // the row's MFMA chain at raised wave priority, its epilogue at the
        // normal one: of the two waves on a SIMD, the one with MFMAs to issue
        // wins the arbiter, so one wave's epilogue runs beside the other's
        // chain (-5 % on the forward kernels)
        __builtin_amdgcn_s_setprio(1);
        Fp = (i + 1 < RPW) ? load_row(in, y0 + i + 1, i + 2 < RPW) : Fe;
        if constexpr (MODE == QTX_CONV_FP32) {
#pragma unroll
          for (int dy = 0; dy < 3; ++dy) {
            const Frag& R = (dy == 0) ? Fm : (dy == 1 ? F0 : Fp);
#pragma unroll
            for (int dx = 0; dx < 3; ++dx)
#pragma unroll
              for (int jp = 0; jp < 4; ++jp)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[(3 * dy + dx) * 4 + jp], R.f[dx][jp], acc, 0, 0, 0);
          }
        } else {
          // taps (dy, 0), (dy, 1): three split products per K-step; tap
          // (dy, 2): [hi | lo] x [X hi; X hi] per dy, then the hi x X lo
          // halves two dy to an instruction (14 MFMAs per row instead of 18)
#pragma unroll
          for (int dy = 0; dy < 3; ++dy) {
            const Frag& R = (dy == 0) ? Fm : (dy == 1 ? F0 : Fp);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wl[2 * dy], R.h[0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wh[2 * dy], R.l[0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wh[2 * dy], R.h[0], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wh[2 * dy + 1], R.h[1], acc, 0, 0, 0);
          }
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wl[1], Fm.l[1], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wl[3], Fp.l[1], acc, 0, 0, 0);
        }
      }
      __builtin_amdgcn_s_setprio(0);
      if (i > 0) epi(i - 1, accp);
      if (i < RPW) {
        accp = acc;
        Fm = F0;
        F0 = Fp;
      }
    }
  };

  char* const buf = act + b * CFGB;  // one activation buffer per configuration, updated in place
  auto layers = [&](auto act_c) {
    constexpr int ACT = decltype(act_c)::value;
    // layers 1 .. 2 nb - 2 in pairs: conv2 of block l / 2 (residual), conv1 of block l / 2 + 1
    for (int l = 1; l < 2 * nb - 1; l += 2) {
      const float scale = rsqrtf((float)(l / 2 + 2));
      constexpr float GA = -2.0f * 0.79788456080286536f * 1.4426950408889634f;
      const float k0 = (ACT == QTX_ACT_GELU_ERF) ? scale * 0.70710678118654752f : scale * GA;
      const float k1 = scale * scale * scale * (GA * 0.044715f);
      run_layer(l, buf, [&](int i, v4f acc) {
        v4f o;
        v4f xr = acc + resr[i];
        resr[i] = xr;
        if constexpr (MODE == QTX_CONV_FP32) {
#pragma unroll
          for (int q = 0; q < 4; ++q) o[q] = act_t<ACT>(xr[q] * scale);
        } else {
          // the next layer's weights carry the scale
#pragma unroll
          for (int q = 0; q < 4; ++q) o[q] = act_over_s<ACT>(xr[q], k0, k1);
        }
        store4(buf + (y0 + i) * ROWB, o);
      });
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      run_layer(l + 1, buf, [&](int i, v4f acc) {
        v4f o;
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = act_t<ACT>(acc[q]);
        store4(buf + (y0 + i) * ROWB, o);
      });
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
  };
  if (actk == QTX_ACT_GELU_ERF) layers(std::integral_constant<int, QTX_ACT_GELU_ERF>{});
  else if (actk == QTX_ACT_RELU) layers(std::integral_constant<int, QTX_ACT_RELU>{});
  else layers(std::integral_constant<int, QTX_ACT_GELU_TANH>{});
  // ---- last layer (conv2 of the last block, no bias, no GELU) and the head
  {
    const int l = 2 * nb - 1;
    const char* in = buf;
    const float scale = rsqrtf((float)(nb + 1));
    // log-sum-exp of the head: each lane keeps a running (max, sum) over its
    // own values of the wave's rows; one wave reduction at the end
    float m_l = -INFINITY, s_l = 0.0f;
    run_layer(l, in, [&](int i, v4f acc) {
      float hv[4];
      const v4f r = resr[i];
#pragma unroll
      for (int q = 0; q < 4; ++q) hv[q] = (acc[q] + r[q]) * scale;
      const float mn = fmaxf(m_l, fmaxf(fmaxf(hv[0], hv[1]), fmaxf(hv[2], hv[3])));
      float sacc = s_l * __expf(m_l - mn);
#pragma unroll
      for (int q = 0; q < 4; ++q) sacc += __expf(hv[q] - mn);
      s_l = sacc;
      m_l = mn;
    });
    const float m_w = wave_max(m_l);
    const float s_w = wave_sum_prod(s_l, __expf(m_l - m_w));
    if (lane == 0) {
      red[wv * 2] = m_w;
      red[wv * 2 + 1] = s_w;
    }
    __syncthreads();
    if (threadIdx.x < B) {
      // merge the four waves' (max, sum) in FP32 (the sums are FP32 already);
      // FP64 exp / log here would hold every wave at the barrier below
      constexpr double kLogCN = 8.317766166719343;  // log(16 channels * 256 sites)
      const int bb = threadIdx.x;
      float m = -INFINITY;
      for (int w = WPC * bb; w < WPC * bb + WPC; ++w) m = fmaxf(m, red[w * 2]);
      float ssum = 0.0f;
      for (int w = WPC * bb; w < WPC * bb + WPC; ++w) ssum += red[w * 2 + 1] * __expf(red[w * 2] - m);
      lp_out[bb] = (double)m + (double)logf(ssum) - kLogCN;
    }
    __syncthreads();
  }
}

// Split-bf16 forward for C = 32 on grids of up to 400 sites (the 20 x 20
// benchmark lattice): one configuration per workgroup of W = 4 waves, two
// workgroups per CU (2 waves per SIMD, at most 256 VGPRs each).  Items are
// 16-site tiles in row-major order; wave w owns tiles w, w + 4, ... (at most
// MAXT = 7 of the 25 of 20 x 20) and computes both 16-channel output tiles
// (CTW = 2) of each, so one B fragment read from LDS feeds six MFMAs.  Per
// layer the K loop runs over the 9 taps outside the tile loop: the A
// fragments of one tap (2 output tiles x hi/lo, 16 VGPRs, prefetched one tap
// ahead from L2) serve every tile of the wave, and the wave's 2 x MAXT
// accumulators are independent MFMA chains.  Activations sit once in LDS
// (bf16 hi/lo, 128 bytes per site, 16-byte chunks XORed with site & 7); a
// layer computes into registers and its outputs replace its inputs between
// two barriers, which halves the LDS of a ping-pong pair so two workgroups
// fit on a CU.  The epilogue runs after the first barrier, one tile at a
// time (GELU, split, store), so the GELU outputs never coexist with the
// accumulators; the next layer's first A fragments are fetched after it.
// That keeps every C = 32 kernel within 256 VGPRs without scratch (GELU
// before the barrier, with all outputs held, spilled 200-370 bytes per lane
// and ran the 20 x 20 sweep at 300 against 378 TFLOP/s).  The B fragment of
// (tap, tile) is found through a table of byte offsets of the tap's source
// site (swizzle key in bits 4-6), built once per launch.  The residual stream
// stays in registers in the MFMA output layout.  CTW = 1 (six waves, wave pairs sharing tiles, three waves per
// SIMD) ran the 20 x 20 sweep at 186-221 TFLOP/s against 301 for CTW = 2:
// it reads every B fragment twice and issues three MFMAs per LDS round trip.
constexpr int RC32_MAXN = 400;
constexpr int RC32_CTW = 2;  // output tiles per wave
constexpr int rc32_tab_bytes(int nmax) { return 9 * nmax * 2; }

template <int MAXT, int W, int CTW, int ACT>
__device__ __attribute__((always_inline)) inline void rc_forward_t32(
    const RcGeom& g, int nb, const char* __restrict__ packed, int64_t off_l0w, int64_t off_l0b,
    int64_t bias_off, int64_t off_frag, int64_t frag_bytes, const int8_t* sp, char* act, const uint16_t* tab,
    float* red, double* lp_out) {
  // CTW output tiles per wave: 1 (wave pairs share tiles, ct = w & 1) or 2
  constexpr int C = 32, NP = (CTW == 1) ? W / 2 : W;  // NP groups of waves own disjoint tiles
  const int lane = threadIdx.x % WAVE;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int gq = lane / 16, x16 = lane % 16;
  const int ct0 = (CTW == 1) ? (wv & 1) : 0, m = (CTW == 1) ? (wv >> 1) : wv;
  const int N = g.N, NT = g.NT;
  const int nti = (NT - m + NP - 1) / NP;  // tiles of this wave (wave-uniform)
  const float* pf = reinterpret_cast<const float*>(packed);
  // the B fragment of lane group gq is chunk gq (hi) / 4 + gq (lo)
  const uint32_t xhi = (uint32_t)gq << 4, xlo = (uint32_t)(gq ^ 4) << 4;
  // output stores: channel 16 ct + 4 gq + i of site p lies in chunk
  // 2 ct + gq / 2 (hi) or 4 + 2 ct + gq / 2 (lo), half gq & 1; the key p & 7
  // equals lane & 7 for every tile (tiles start at multiples of 16)
  const int key = lane & 7;
  int st_hi[CTW], st_lo[CTW];
#pragma unroll
  for (int j = 0; j < CTW; ++j) {
    const int ct = ct0 + j;
    st_hi[j] = x16 * 128 + (((2 * ct + (gq >> 1)) ^ key) << 4) + (gq & 1) * 8;
    st_lo[j] = x16 * 128 + (((4 + 2 * ct + (gq >> 1)) ^ key) << 4) + (gq & 1) * 8;
  }
  auto site = [&](int k) { return 16 * (m + NP * k) + x16; };  // may be >= N
  auto store4 = [&](int k, int j, v4f v) {
    const int t = m + NP * k;
    if (16 * t + x16 < N) {
      v4bf hi, lo;
      split_bf16x4(v, hi, lo);
      char* base = act + t * 16 * 128;
      *reinterpret_cast<v4bf*>(base + st_hi[j]) = hi;
      *reinterpret_cast<v4bf*>(base + st_lo[j]) = lo;
    }
  };
  // A fragments (hi, lo) of (layer, tap) for this wave's output tiles
  auto load_a = [&](int l, int ks, v8bf (&a)[CTW][2]) {
#pragma unroll
    for (int j = 0; j < CTW; ++j) {
      const v8bf* q = reinterpret_cast<const v8bf*>(packed + off_frag + (int64_t)l * frag_bytes) +
                      (((ct0 + j) * 9 + ks) * WAVE + lane) * 2;
      a[j][0] = q[0];
      a[j][1] = q[1];
    }
  };

  v4f res[MAXT][CTW];

  // ---- layer 0: conv (Cin = 1) of s / sqrt(2) on VALU, GELU, into act
  {
    // this lane's 4 CTW output channels: weights co * 9 + tap from one base
    const float* W0 = pf + off_l0w + (16 * ct0 + 4 * gq) * 9;
    const float* b0 = pf + off_l0b + 16 * ct0 + 4 * gq;
#pragma unroll
    for (int k = 0; k < MAXT; ++k) {
      if (k < nti) {
        const int p = site(k);
        const int pc = p < N ? p : N - 1;
        float sv[9];
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) sv[tap] = (float)sp[tab[tap * RC32_MAXN + pc] >> 7] * 0.70710678118654752f;
        const float spin = (float)sp[pc];
#pragma unroll
        for (int j = 0; j < CTW; ++j) {
          v4f z;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int co = 16 * j + q;
            float a = b0[co];
#pragma unroll
            for (int tap = 0; tap < 9; ++tap) a += W0[co * 9 + tap] * sv[tap];
            z[q] = act_t<ACT>(a);
          }
          res[k][j] = v4f{spin, spin, spin, spin};
          store4(k, j, z);
        }
      }
    }
  }
  v8bf an[CTW][2];
  load_a(1, 0, an);
  __syncthreads();

  for (int l = 1; l < 2 * nb; ++l) {
    const float* bias = pf + bias_off + (int64_t)l * C;
    v4f acc[MAXT][CTW];
#pragma unroll
    for (int j = 0; j < CTW; ++j) {
      const int cb = 16 * (ct0 + j) + 4 * gq;
      const v4f b4 = v4f{bias[cb], bias[cb + 1], bias[cb + 2], bias[cb + 3]};
#pragma unroll
      for (int k = 0; k < MAXT; ++k) acc[k][j] = b4;
    }
    const bool last = (l == 2 * nb - 1);
    // the tap offsets are the same in every layer: an opaque per-layer zero
    // keeps the compiler from hoisting all 9 x MAXT of them out of the layer
    // loop into registers
    int tz = 0;
    asm volatile("" : "+s"(tz));
    // the layer's MFMA loop at raised wave priority, the epilogue at the
    // normal one, so that the other workgroup's epilogue runs beside it
    __builtin_amdgcn_s_setprio(1);
#pragma unroll 1
    for (int ks = 0; ks < 9; ++ks) {
      v8bf a[CTW][2];
#pragma unroll
      for (int j = 0; j < CTW; ++j) {
        a[j][0] = an[j][0];
        a[j][1] = an[j][1];
      }
      if (ks < 8) load_a(l, ks + 1, an);
      const uint16_t* tk = tab + ks * RC32_MAXN + tz;
      // tiles that exist for every wave run unconditionally (sites past N
      // read the table's padding, offset 0, and are never stored); only the
      // last is guarded
#pragma unroll
      for (int k = 0; k < MAXT; ++k) {
        if (k < MAXT - 1 || k < nti) {
          const uint32_t off = tk[site(k)];  // < RC32_MAXN for every tile read here
          const v8bf bh = *reinterpret_cast<const v8bf*>(act + (off ^ xhi));
          const v8bf bl = *reinterpret_cast<const v8bf*>(act + (off ^ xlo));
#pragma unroll
          for (int j = 0; j < CTW; ++j) {
            acc[k][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j][1], bh, acc[k][j], 0, 0, 0);
            acc[k][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j][0], bl, acc[k][j], 0, 0, 0);
            acc[k][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j][0], bh, acc[k][j], 0, 0, 0);
          }
        }
      }
    }
    __builtin_amdgcn_s_setprio(0);
    if (!last) {
      const bool is_conv2 = (l % 2) == 1;
      const float scale = is_conv2 ? rsqrtf((float)(l / 2 + 2)) : 1.0f;
      __syncthreads();  // every wave has read this layer's input
#pragma unroll
      for (int k = 0; k < MAXT; ++k) {
        if (k < nti) {
#pragma unroll
          for (int j = 0; j < CTW; ++j) {
            v4f o;
            if (is_conv2) {
              const v4f xr = acc[k][j] + res[k][j];
              res[k][j] = xr;
#pragma unroll
              for (int q = 0; q < 4; ++q) o[q] = act_t<ACT>(xr[q] * scale);
            } else {
#pragma unroll
              for (int q = 0; q < 4; ++q) o[q] = act_t<ACT>(acc[k][j][q]);
            }
            store4(k, j, o);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      load_a(l + 1, 0, an);
      __syncthreads();
    } else {
      // head: h = (z2 + r) / sqrt(nb + 1); per-lane running logsumexp, one
      // wave reduction, then the waves' (max, sum) merged in FP32
      const float scale = rsqrtf((float)(nb + 1));
      float m_l = -INFINITY, s_l = 0.0f;
#pragma unroll
      for (int k = 0; k < MAXT; ++k) {
        if (k >= nti || site(k) >= N) continue;
#pragma unroll
        for (int j = 0; j < CTW; ++j) {
          float hv[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) hv[q] = (acc[k][j][q] + res[k][j][q]) * scale;
          const float mn = fmaxf(m_l, fmaxf(fmaxf(hv[0], hv[1]), fmaxf(hv[2], hv[3])));
          float sacc = s_l * __expf(m_l - mn);
#pragma unroll
          for (int q = 0; q < 4; ++q) sacc += __expf(hv[q] - mn);
          s_l = sacc;
          m_l = mn;
        }
      }
      const float m_w = wave_max(m_l);
      const float s_w = wave_sum(m_l > -INFINITY ? s_l * __expf(m_l - m_w) : 0.0f);
      if (lane == 0) {
        red[wv * 2] = m_w;
        red[wv * 2 + 1] = s_w;
      }
      __syncthreads();
      if (threadIdx.x == 0) {
        float mx = -INFINITY;
        for (int w = 0; w < W; ++w) mx = fmaxf(mx, red[w * 2]);
        float ssum = 0.0f;
        for (int w = 0; w < W; ++w)
          if (red[w * 2] > -INFINITY) ssum += red[w * 2 + 1] * __expf(red[w * 2] - mx);
        lp_out[0] = (double)mx + (double)logf(ssum) - g.log_cn;
      }
      __syncthreads();
    }
  }
}

// byte offsets (source site * 128 | (source site & 7) << 4) of the 9 taps of
// every site, tab[tap * RC32_MAXN + p], padded with offset 0 up to
// RC32_MAXN sites; all threads of the block call it
__device__ __forceinline__ void rc32_build_tab(const RcGeom& g, uint16_t* tab) {
  for (int e = threadIdx.x; e < 9 * RC32_MAXN; e += blockDim.x) {
    const int tap = e / RC32_MAXN, p = e - tap * RC32_MAXN;
    uint16_t v = 0;
    if (p < g.N) {
      const int src = tap_pos(g, p / g.L1, p % g.L1, tap);
      v = (uint16_t)((src << 7) | ((src & 7) << 4));
    }
    tab[e] = v;
  }
}

// ---------------------------------------------------------------- kernels
#define RC_FWD(SP, LP)                                                                                        \
  do {                                                                                                        \
    if constexpr (ROWS == 3) {                                                                                \
      const uint16_t* tab_ = reinterpret_cast<const uint16_t*>(wst);                                          \
      if (a.actk == QTX_ACT_GELU_ERF)                                                                         \
        rc_forward_t32<MAXT, W, RC32_CTW, QTX_ACT_GELU_ERF>(a.g, a.nb, a.packed, a.off_l0w, a.off_l0b,         \
                                                            a.bias_off, a.off_frag, a.frag_bytes, SP, act,     \
                                                            tab_, red, LP);                                    \
      else if (a.actk == QTX_ACT_RELU)                                                                        \
        rc_forward_t32<MAXT, W, RC32_CTW, QTX_ACT_RELU>(a.g, a.nb, a.packed, a.off_l0w, a.off_l0b, a.bias_off, \
                                                        a.off_frag, a.frag_bytes, SP, act, tab_, red, LP);     \
      else                                                                                                    \
        rc_forward_t32<MAXT, W, RC32_CTW, QTX_ACT_GELU_TANH>(a.g, a.nb, a.packed, a.off_l0w, a.off_l0b,        \
                                                             a.bias_off, a.off_frag, a.frag_bytes, SP, act,    \
                                                             tab_, red, LP);                                   \
    } else                                                                                                    \
      rc_forward_win<MODE, B, W / B>(a.g, a.nb, a.actk, a.packed, a.off_l0w, a.off_l0b, a.bias_off, a.off_frag, \
                           a.frag_bytes, SP, act, wst, red, LP);                                              \
  } while (0)

template <int C, int MODE, int B, int NMAX, int MAXT, int W, int ROWS>
__global__ __launch_bounds__(W * 64, 2) void rc_logpsi_kernel(RcArgs a, const int8_t* __restrict__ s, int64_t ns,
                                                               double* __restrict__ logabs) {
  __shared__ __attribute__((aligned(16))) char act[B * NMAX * C * 4];
  __shared__ __attribute__((aligned(16))) char wst[ROWS == 2 ? rc_win_lds(B) : rc32_tab_bytes(NMAX)];
  __shared__ int8_t sp[B * NMAX];
  __shared__ float red[2 * B * W];
  __shared__ double lp[B];
  const int N = a.g.N;
  const int64_t c0 = xcd_block(blockIdx.x, gridDim.x) * B;  // per-chain Philox words of a step share lines
  for (int i = threadIdx.x; i < B * N; i += (W * WAVE)) {
    int b = i / N;
    sp[i] = (c0 + b < ns) ? s[(c0 + b) * N + (i % N)] : (int8_t)1;
  }
  if constexpr (ROWS == 3) rc32_build_tab(a.g, reinterpret_cast<uint16_t*>(wst));
  __syncthreads();
  RC_FWD(sp, lp);
  if (threadIdx.x < B && c0 + threadIdx.x < ns) logabs[c0 + threadIdx.x] = lp[threadIdx.x];
}

template <int C, int MODE, int B, int NMAX, int MAXT, int W, int ROWS>
__global__ __launch_bounds__(W * 64, 2) void rc_metropolis_kernel(
    RcArgs a, int kind, const int32_t* __restrict__ nbr, int width, int hopping, const uint32_t* __restrict__ words,
    int nsteps, int64_t ns, double reweight, double tie_tol, int8_t* __restrict__ s, double* __restrict__ logabs,
    int32_t* __restrict__ n_accept, int32_t* __restrict__ n_near) {
  __shared__ __attribute__((aligned(16))) char act[B * NMAX * C * 4];
  __shared__ __attribute__((aligned(16))) char wst[ROWS == 2 ? rc_win_lds(B) : rc32_tab_bytes(NMAX)];
  __shared__ int8_t cur[B * NMAX];
  __shared__ int8_t prop[B * NMAX];
  __shared__ float red[2 * B * W];
  __shared__ double lp_new[B];
  __shared__ double lp_cur[B];
  __shared__ int mv_a[B], mv_b[B], mv_upd[B], nhop[B], nacc[B], nnear[B];
  __shared__ double mv_thr[B];
  __shared__ uint2 wq[B][WAVE];   // proposal words of 64 steps
  __shared__ double tq[B][WAVE];  // and their acceptance thresholds
  const int N = a.g.N;
  const int lane = threadIdx.x % WAVE, wv = threadIdx.x / WAVE;
  const int64_t c0 = xcd_block(blockIdx.x, gridDim.x) * B;  // per-chain Philox words of a step share lines
  for (int i = threadIdx.x; i < B * N; i += (W * WAVE)) {
    int b = i / N;
    cur[i] = (c0 + b < ns) ? s[(c0 + b) * N + (i % N)] : (int8_t)1;
  }
  if (threadIdx.x < B) {
    int b = threadIdx.x;
    lp_cur[b] = (c0 + b < ns) ? logabs[c0 + b] : 0.0;
    nacc[b] = 0;
    nnear[b] = 0;
  }
  if constexpr (ROWS == 3) rc32_build_tab(a.g, reinterpret_cast<uint16_t*>(wst));
  __syncthreads();
  for (int b = wv; b < B; b += W) {
    int cnt = 0;
    for (int i = lane; i < N; i += WAVE) cnt += (cur[b * N + i] == hopping);
    cnt = wave_sum(cnt);
    if (lane == 0) nhop[b] = cnt;
  }
  __syncthreads();
  static_assert(W >= B, "one wave per chain at most");
  // A proposal that leaves the spins unchanged (an exchange of equal spins: a
  // third to a half of them at Sz = 0) is never accepted, so its forward is
  // not run: wave b < B draws chain b's moves until one changes the spins, and
  // the chains of a workgroup may be at different steps.  The Philox words of
  // 64 steps are fetched at once, lane l step t0 + l, and each lane evaluates
  // its step's FP64 threshold.  512 steps of 4096 chains, 16 x 16, 8 blocks:
  // 104.6 -> 57.3 ms.
  int tc = 0;  // next step of the wave's chain
  for (;;) {
    // the lane index through an opaque move, as in the forwards: the step's
    // per-lane LDS addresses are formed here, not held across the loop
    int lane = threadIdx.x % WAVE;
    asm volatile("" : "+v"(lane));
    if (wv < B) {
      const int b = wv;
      const int64_t c = c0 + b;
      int fa = -1, fb = -1;
      bool upd = false;
      double thr = 0.0;
      while (c < ns && tc < nsteps && !upd) {
        const int q = tc % WAVE;
        if (q == 0) {
          if (tc + lane < nsteps) {
            const uint4 w = reinterpret_cast<const uint4*>(words)[(int64_t)(tc + lane) * ns + c];
            wq[b][lane] = make_uint2(w.x, w.y);
            tq[b][lane] = accept_threshold(w.z, w.w);
          }
          wave_lds_fence();
        }
        const uint2 w = wq[b][q];
        propose_move(kind, cur + b * N, N, nbr, width, hopping, nhop[b], w.x, w.y, lane, fa, fb, upd);
        thr = tq[b][q];
        ++tc;
      }
      for (int i = lane; i < N; i += WAVE) {
        int8_t v = cur[b * N + i];
        if (upd && (i == fa || i == fb)) v = -v;
        prop[b * N + i] = v;
      }
      if (lane == 0) {
        mv_a[b] = fa;
        mv_b[b] = fb;
        mv_upd[b] = upd ? 1 : 0;
        mv_thr[b] = thr;
      }
    }
    __syncthreads();
    int any = 0;
#pragma unroll
    for (int b = 0; b < B; ++b) any |= mv_upd[b];
    if (!any) break;  // every chain has run its steps
    RC_FWD(prop, lp_new);
    // accept / reject (rc_forward ends with a barrier)
    for (int b = wv; b < B; b += W) {
      if (!mv_upd[b]) continue;
      double d = reweight * (lp_new[b] - lp_cur[b]);
      double thr = mv_thr[b];
      bool acc = (d > thr) || (lp_cur[b] == -INFINITY);
      if (acc) {
        int fa = mv_a[b], fb = mv_b[b];
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) {
          cur[b * N + fa] = -cur[b * N + fa];
          if (fb >= 0) cur[b * N + fb] = -cur[b * N + fb];
          lp_cur[b] = lp_new[b];
          nacc[b] += 1;
        }
      }
      if (lane == 0 && fabs(d - thr) < tie_tol) nnear[b] += 1;
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < B * N; i += (W * WAVE)) {
    int b = i / N;
    if (c0 + b < ns) s[(c0 + b) * N + (i % N)] = cur[i];
  }
  if (threadIdx.x < B && c0 + threadIdx.x < ns) {
    int b = threadIdx.x;
    logabs[c0 + b] = lp_cur[b];
    n_accept[c0 + b] += nacc[b];
    n_near[c0 + b] += nnear[b];
  }
}

constexpr int RC_MAXCAND = 4096;
constexpr int RC_MAXCAND_WIN = 3072;  // 16 x 16 window kernels: keeps two workgroups' LDS within a CU

template <int C, int MODE, int B, int NMAX, int MAXT, int W, int ROWS>
__global__ __launch_bounds__(W * 64, 2) void rc_eloc_kernel(RcArgs a, qtx_ham H, const int8_t* __restrict__ s,
                                                             const double* __restrict__ logabs, int S,
                                                             double* __restrict__ eloc, int32_t* __restrict__ nconn) {
  // S workgroups per sample (virtual block n S + sp): workgroup sp evaluates
  // the sp-th of S near-equal runs of candidates into eloc[n S + sp] (partial
  // sums for rc_eloc_sum_kernel when S > 1, the local energy when S = 1)
  __shared__ __attribute__((aligned(16))) char act[B * NMAX * C * 4];
  __shared__ __attribute__((aligned(16))) char wst[ROWS == 2 ? rc_win_lds(B) : rc32_tab_bytes(NMAX)];
  __shared__ int8_t s0[NMAX];
  __shared__ int8_t prop[B * NMAX];
  __shared__ float red[2 * B * W];
  __shared__ double lp[B];
  __shared__ int16_t vlist[ROWS == 2 ? RC_MAXCAND_WIN : RC_MAXCAND];
  __shared__ int nvalid_s;
  __shared__ double diag_s, e_s;
  __shared__ int16_t mv[4 * B];  // slot b: flips applied (2), flips of the next candidate (2)
  const int N = a.g.N;
  const int lane = threadIdx.x % WAVE, wv = threadIdx.x / WAVE;
  const int64_t n = blockIdx.x / (unsigned)S;
  const int sp = (int)(blockIdx.x % (unsigned)S);
  for (int i = threadIdx.x; i < N; i += (W * WAVE)) s0[i] = s[n * N + i];
  if constexpr (ROWS == 3) rc32_build_tab(a.g, reinterpret_cast<uint16_t*>(wst));
  __syncthreads();
  if (wv == 0) {
    // diagonal part and the ordered list of valid candidates (ballot compaction)
    double dg = diag_energy(H, s0, lane);
    int pos = 0;
    for (int base = 0; base < H.noff; base += WAVE) {
      int k = base + lane;
      bool v = (k < H.noff) && cand_valid(H, s0, k);
      uint64_t m = __ballot(v);
      uint64_t below = (lane == 0) ? 0ull : (m & ((~0ull) >> (64 - lane)));
      if (v) vlist[pos + __popcll(below)] = (int16_t)k;
      pos += __popcll(m);
    }
    if (lane == 0) {
      nvalid_s = pos;
      diag_s = dg;
    }
  }
  __syncthreads();
  const int nall = nvalid_s;
  // runs start at multiples of B candidates
  const int nbatch = (nall + B - 1) / B;
  const int first = (int)((int64_t)nbatch * sp / S) * B;
  const int last = (int)((int64_t)nbatch * (sp + 1) / S) * B;
  const int nvalid = last < nall ? last : nall;  // end of this workgroup's run
  const double lp0 = logabs[n];
  // prop[b] holds s0 with candidate start + b applied: thread b < B undoes
  // the previous candidate's (at most two) flips and applies the next one's,
  // whose sites were fetched before the forward.  These flips and the sum
  // live in LDS, not in registers held across the forward.
  for (int i = threadIdx.x; i < B * N; i += (W * WAVE)) prop[i] = s0[i % N];
  if (threadIdx.x < B) {
    const int b = threadIdx.x;
    int na = -1, nb = -1;
    if (first + b < nvalid) {
      const int k = vlist[first + b];
      na = H.off_a[k];
      nb = H.off_b[k];
    }
    mv[4 * b] = (int16_t)na;
    mv[4 * b + 1] = (int16_t)nb;
  }
  if (threadIdx.x == 0) e_s = 0.0;
  __syncthreads();
  if (threadIdx.x < B) {
    const int b = threadIdx.x;
    int8_t* pb = prop + b * N;
    const int na = mv[4 * b], nb = mv[4 * b + 1];
    if (na >= 0) pb[na] = -s0[na];
    if (nb >= 0) pb[nb] = -s0[nb];
  }
  __syncthreads();
  for (int start = first; start < nvalid; start += B) {
    // thread b < B: the next candidate's sites and this candidate's coupling,
    // fetched before the forward and held in registers across it (their
    // global-memory latency hidden by the forward)
    int na = -1, nb = -1;
    double cb = 0.0;
    if (threadIdx.x < B) {
      const int b = threadIdx.x;
      if (start + B + b < nvalid) {
        const int k = vlist[start + B + b];
        na = H.off_a[k];
        nb = H.off_b[k];
      }
      if (start + b < nvalid) cb = H.off_c[vlist[start + b]];
    }
    RC_FWD(prop, lp);
    if (wv == 0) {
      // sum in candidate order by thread 0, as the couplings' owners pass them on
      double term = 0.0;
      if (lane < B && start + lane < nvalid) term = cb * exp_ratio(lp[lane] - lp0);
      double e = e_s;
      for (int b = 0; b < B && start + b < nvalid; ++b) e += __shfl(term, b);
      if (lane == 0) e_s = e;
    }
    if (threadIdx.x < B) {
      const int b = threadIdx.x;
      int8_t* pb = prop + b * N;
      const int fa = mv[4 * b], fb = mv[4 * b + 1];
      if (fa >= 0) pb[fa] = s0[fa];
      if (fb >= 0) pb[fb] = s0[fb];
      if (na >= 0) pb[na] = -s0[na];
      if (nb >= 0) pb[nb] = -s0[nb];
      mv[4 * b] = (int16_t)na;
      mv[4 * b + 1] = (int16_t)nb;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    eloc[blockIdx.x] = (sp == 0) ? diag_s + e_s : e_s;
    if (nconn && sp == 0) nconn[n] = nall;
  }
}
#undef RC_FWD

// eloc[n] = sum of sample n's S partial sums, in order
__global__ void rc_eloc_sum_kernel(const double* __restrict__ part, int64_t ns, int S, double* __restrict__ eloc) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= ns) return;
  double e = 0.0;
  for (int sp = 0; sp < S; ++sp) e += part[n * S + sp];
  eloc[n] = e;
}


}  // namespace qtx

using namespace qtx;

// ================================================================ C ABI
static RcArgs rc_args(const RcLayout& L, const void* packed) {
  RcArgs a;
  a.g = RcGeom{L.L0, L.L1, L.N, (L.N + 15) / 16, std::log((double)L.C * (double)L.N)};
  a.nb = L.nb;
  a.actk = L.actk;
  a.packed = (const char*)packed;
  a.off_l0w = L.off_l0w;
  a.off_l0b = L.off_l0b;
  a.bias_off = L.bias_off;
  a.off_frag = L.off_frag;
  a.frag_bytes = L.frag_bytes;
  a.off_jac = L.off_jac;
  return a;
}

// The 16 x 16 window kernels (two configurations per workgroup) and the large
// 32-channel split-bf16 ones (one); every other shape runs the kernels of
// resconv_wave.hpp
static bool rc_own_kernel(const RcLayout& L) {
  return L.win || (L.C == 32 && L.mode == QTX_CONV_BF16X3 && (L.N + 15) / 16 > 16);
}

#define RC_DISPATCH(KERNEL, GRID_FROM_B, ...)                                                          \
  do {                                                                                                 \
    if (L.win) {                                                                                       \
      constexpr int B_ = 2;                                                                            \
      dim3 grid_ = GRID_FROM_B;                                                                        \
      if (L.mode == QTX_CONV_FP32)                                                                     \
        hipLaunchKernelGGL((KERNEL<16, QTX_CONV_FP32, 2, 256, 4, 4, 2>), grid_, dim3(256), 0, st, __VA_ARGS__); \
      else                                                                                             \
        hipLaunchKernelGGL((KERNEL<16, QTX_CONV_BF16X3, 2, 256, 4, 4, 2>), grid_, dim3(256), 0, st, __VA_ARGS__); \
    } else {                                                                                           \
      constexpr int B_ = 1;                                                                            \
      dim3 grid_ = GRID_FROM_B;                                                                        \
      hipLaunchKernelGGL((KERNEL<32, QTX_CONV_BF16X3, 1, RC32_MAXN, 7, 4, 3>), grid_, dim3(256), 0, st, __VA_ARGS__); \
    }                                                                                                  \
  } while (0)

extern "C" {

int64_t qtx_resconv_nparams(const qtx_resconv_desc* d) {
  if (!d || d->nblocks < 1 || d->channels < 1) return -1;
  return rc_nparams(d->nblocks, d->channels);
}

size_t qtx_resconv_packed_bytes(const qtx_resconv_desc* d) {
  if (rc_check(d) != QTX_OK) return 0;
  return (size_t)rc_layout(d).total_bytes;
}

int qtx_resconv_pack(void* stream, const qtx_resconv_desc* d, const float* theta, void* packed) {
  int rc = rc_check(d);
  if (rc) return rc;
  QTX_REQUIRE(theta && packed, "null pointer");
  RcLayout L = rc_layout(d);
  hipStream_t st = as_stream(stream);
  const int64_t n = L.nparams + (int64_t)L.C * 10 + (int64_t)2 * L.nb * L.C + (int64_t)(2 * L.nb - 1) * 2 * L.C * L.C * 9;
  float* frag = (float*)((char*)packed + L.off_jac);
  const dim3 b(256), gp((unsigned)((n + 255) / 256));
  if (L.C == 16)
    hipLaunchKernelGGL(rc_pack_kernel<16>, gp, b, 0, st, theta, L.nb, L.nparams, (float*)packed, L.off_l0w, L.off_l0b,
                       L.bias_off, frag);
  else
    hipLaunchKernelGGL(rc_pack_kernel<32>, gp, b, 0, st, theta, L.nb, L.nparams, (float*)packed, L.off_l0w, L.off_l0b,
                       L.bias_off, frag);
  if (L.frag_bytes > 0) {
    const dim3 g((unsigned)((rc_frag_steps(L) * WAVE * (2 * L.nb - 1) + 255) / 256));
    if (L.mode == QTX_CONV_FP32)
      hipLaunchKernelGGL((rc_pack_frag_kernel<16, QTX_CONV_FP32, 1>), g, b, 0, st, theta, L.nb, (char*)packed,
                         L.off_frag, L.frag_bytes);
    else if (L.win)
      hipLaunchKernelGGL((rc_pack_frag_kernel<16, QTX_CONV_BF16X3, 1>), g, b, 0, st, theta, L.nb, (char*)packed,
                         L.off_frag, L.frag_bytes);
    else if (L.C == 16)
      hipLaunchKernelGGL((rc_pack_frag_kernel<16, QTX_CONV_BF16X3, 0>), g, b, 0, st, theta, L.nb, (char*)packed,
                         L.off_frag, L.frag_bytes);
    else
      hipLaunchKernelGGL((rc_pack_frag_kernel<32, QTX_CONV_BF16X3, 0>), g, b, 0, st, theta, L.nb, (char*)packed,
                         L.off_frag, L.frag_bytes);
  }
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

int qtx_resconv_logpsi(void* stream, const qtx_resconv_desc* d, const void* packed, const int8_t* s, int64_t ns,
                       double* logabs) {
  int rc = rc_check(d);
  if (rc) return rc;
  QTX_REQUIRE(packed && ns >= 0 && (ns == 0 || (s && logabs)), "bad arguments");
  if (ns == 0) return QTX_OK;
  RcLayout L = rc_layout(d);
  RcArgs a = rc_args(L, packed);
  hipStream_t st = as_stream(stream);
  if (!rc_own_kernel(L))
    return RW_CALL(rw_logpsi, L, st, L, a, s, ns, logabs);
  RC_DISPATCH(rc_logpsi_kernel, dim3((unsigned)((ns + B_ - 1) / B_)), a, s, ns, logabs);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

int qtx_resconv_metropolis(void* stream, const qtx_resconv_desc* d, const void* packed, int kind,
                           const int32_t* nbr, int32_t width, int32_t hopping, const uint32_t* words,
                           int32_t nsteps, int64_t ns, double reweight, double tie_tol, int8_t* s, double* logabs,
                           int32_t* n_accept, int32_t* n_near) {
  int rc = rc_check(d);
  if (rc) return rc;
  QTX_REQUIRE(kind == QTX_LOCALFLIP || kind == QTX_EXCHANGE, "kind must be QTX_LOCALFLIP or QTX_EXCHANGE");
  QTX_REQUIRE(kind == QTX_LOCALFLIP || (nbr != nullptr && width > 0), "EXCHANGE needs a neighbour table");
  QTX_REQUIRE(hopping == 1 || hopping == -1, "hopping must be +1 or -1");
  QTX_REQUIRE(nsteps >= 0 && ns >= 0, "negative size");
  QTX_REQUIRE(packed && (ns == 0 || (s && logabs && n_accept && n_near && (nsteps == 0 || words))),
              "null pointer");
  if (ns == 0) return QTX_OK;
  RcLayout L = rc_layout(d);
  RcArgs a = rc_args(L, packed);
  hipStream_t st = as_stream(stream);
  if (!rc_own_kernel(L))
    return RW_CALL(rw_metropolis, L, st, L, a, kind, nbr, width, hopping, words, nsteps, ns, reweight, tie_tol, s,
                   logabs, n_accept, n_near);
  RC_DISPATCH(rc_metropolis_kernel, dim3((unsigned)((ns + B_ - 1) / B_)), a, kind, nbr, width, hopping, words,
              nsteps, ns, reweight, tie_tol, s, logabs, n_accept, n_near);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

// Workgroups per sample of an E_loc launch.  One workgroup takes a sample's
// candidates one batch after another, so a launch of few samples leaves the
// card's 512 slots (256 CUs, two workgroups each) idle and one of a few
// rounds ends in a nearly empty round: the candidates are split until the
// launch has about 16 rounds, in runs of at least 8 batches (the scan that
// lists a sample's candidates costs each workgroup about as much as one
// forward of a small network).  A quarter of the table is the valid share of
// an exchange Hamiltonian at Sz = 0; with a larger share the runs are longer.
// Measured on J1-J2: 128 samples of 20 x 20, 32 channels, 16 blocks 219.6 ->
// 65.3 ms; 2048 samples of 16 x 16, 8 blocks 53.2 -> 51.3 ms; 1000 samples of
// 10 x 10, 4 blocks (FP32) 17.6 -> 17.0 ms.
static int eloc_split(const RcLayout& L, int32_t noff, int64_t ns) {
  const int64_t want = (16 * 512 + ns - 1) / ns;
  const int batch = L.win ? 2 : (rc_own_kernel(L) ? 1 : 4 / rw_eloc_pick(L.C, L.N, noff, ns).P);
  const int64_t most = noff / 4 / (8 * batch);
  return (int)std::max<int64_t>(1, std::min(want, most));
}

size_t qtx_resconv_eloc_ws_bytes(const qtx_resconv_desc* d, const qtx_ham* H, int64_t ns) {
  if (rc_check(d) != QTX_OK || H == nullptr || H->noff < 0 || ns <= 0) return 0;
  const int S = eloc_split(rc_layout(d), H->noff, ns);
  return S > 1 ? (size_t)ns * S * sizeof(double) : 0;
}

int qtx_resconv_eloc_ws(void* stream, const qtx_resconv_desc* d, const void* packed, const qtx_ham* H,
                        const int8_t* s, const double* logabs, int64_t ns, double* eloc, int32_t* nconn, void* ws,
                        size_t ws_bytes) {
  int rc = rc_check(d);
  if (rc) return rc;
  QTX_REQUIRE(H != nullptr, "null qtx_ham");
  QTX_REQUIRE(H->N == d->L0 * d->L1, "qtx_ham.N != L0 * L1");
  RcLayout L = rc_layout(d);
  QTX_REQUIRE(H->noff <= (L.win ? RC_MAXCAND_WIN : RC_MAXCAND),
              L.win ? "too many off-diagonal candidates (max 3072 on a 16 x 16 lattice with 16 channels)"
                    : "too many off-diagonal candidates (max 4096)");
  QTX_REQUIRE(H->noff == 0 || (H->off_a && H->off_b && H->off_ra && H->off_rb && H->off_c), "null table");
  QTX_REQUIRE(H->ndiag == 0 || (H->diag_c && H->diag_a && H->diag_b && H->diag_kind), "null table");
  QTX_REQUIRE(packed && ns >= 0 && (ns == 0 || (s && logabs && eloc)), "bad arguments");
  if (ns == 0) return QTX_OK;
  QTX_REQUIRE(ns <= 0x7fffffff, "ns too large");
  int S = 1;
  if (ws != nullptr) {
    S = eloc_split(L, H->noff, ns);
    const size_t need = S > 1 ? (size_t)ns * S * sizeof(double) : 0;
    if (ws_bytes < need)
      return fail(QTX_EWORKSPACE, "workspace too small: need " + std::to_string(need) + " bytes");
  }
  RcArgs a = rc_args(L, packed);
  hipStream_t st = as_stream(stream);
  double* out = S > 1 ? (double*)ws : eloc;
  if (rc_own_kernel(L))
    RC_DISPATCH(rc_eloc_kernel, dim3((unsigned)(ns * S)), a, *H, s, logabs, S, out, nconn);
  else if ((rc = RW_CALL(rw_eloc, L, st, L, a, *H, s, logabs, ns, S, out, nconn)))
    return rc;
  if (S > 1)
    hipLaunchKernelGGL(rc_eloc_sum_kernel, dim3((unsigned)((ns + 255) / 256)), dim3(256), 0, st, out, ns, S, eloc);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

int qtx_resconv_eloc(void* stream, const qtx_resconv_desc* d, const void* packed, const qtx_ham* H,
                     const int8_t* s, const double* logabs, int64_t ns, double* eloc, int32_t* nconn) {
  return qtx_resconv_eloc_ws(stream, d, packed, H, s, logabs, ns, eloc, nconn, nullptr, 0);
}

}  // extern "C"
