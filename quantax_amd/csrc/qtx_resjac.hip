// Per-sample log-derivatives of ResConv: forward recompute, backward pass and
// the weight gradients as FP32-MFMA GEMMs, one workgroup per sample.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>

#include "resconv.hpp"

namespace qtx {

// ---------------------------------------------------------------- Jacobian
// One workgroup (4 waves) per sample, persistent over samples.  Every
// convolution of the forward recompute and of the backward pass is an
// FP32-MFMA GEMM (16x16x4 f32) over position-major activations in LDS:
//   forward     Z[co][p]       = sum_{ci,tap} W[co][ci][tap] X[nb(p, tap)][ci]
//   input grad  dX[ci][q]      = sum_{co,tap} W[co][ci][tap] dZ[nb(q, 8 - tap)][co]
//   weight grad G[co][ci,tap]  = sum_p dZ[p][co] X[nb(p, tap)][ci]
// (MFMA lane l holds A[m0 + l%16][k0 + l/16], B[k0 + l/16][n0 + l%16]; result
// element i of lane l is D[m0 + 4(l/16) + i][n0 + l%16].)  The first two are
// the same routine on two sets of packed fragments: a lane reads four
// channels of a tap's source position in one ds_read_b128 and feeds four
// MFMAs.  The weight gradient has K = positions: 16 lanes read the 16
// channels of one position (64 bytes in a row), one ds_read_b32 per MFMA, the
// A operand shared by the nine taps; the waves split the positions (and, with
// 32 channels, the output tiles) and add their accumulators through LDS in a
// fixed order.  Residual stream and running gradient stay in registers in the
// MFMA output layout.  The forward records only x_i and z1_i (conv1's output)
// per block -- the activations are formed again -- lane by lane in that same
// layout, in a slot per workgroup that stays in the memory-side cache.
// Bound: FP32 MFMA (3 F per sample); 16 x 16, 16 channels, 8 blocks, 4096
// samples: 8.55 -> 2.62 ms, 83 TFLOP/s (channel-major operands gathered lane by lane
// through a neighbour table before, and four records per block through HBM).
constexpr int JAC_THREADS = 256;

constexpr int JAC_SLOTS = 768;  // workgroups of a launch: three per CU

struct JacLds {  // byte offsets in the workgroup's dynamic LDS
  int bufb;      // one activation buffer
  int tabc, tabp, spf, sred, total;
};

template <int C>
__host__ __device__ inline JacLds jac_lds(int N) {
  constexpr int CT = C / 16, P = 4 / CT;
  JacLds L;
  const int npad = (N + 15) / 16 * 16;
  L.bufb = npad * C * 4;
  // the two buffers, reused by the weight gradient's sums: (P - 1) parts of
  // every 16 x 16 block, then the summed blocks
  const int red = CT * 9 * CT * 1024 * P;
  int off = 2 * L.bufb > red ? 2 * L.bufb : red;
  L.tabc = off;  // [9][npad] uint16: byte offset of the tap's source position, swizzle key in place
  off += 9 * npad * 2;
  L.tabp = off;  // [npad][16] uint16: the same by position, nine entries used
  off += npad * 32;
  L.spf = off;   // the sample's spins as floats
  off += npad * 4;
  L.sred = off;  // small reductions: 4 x C floats
  off += 4 * C * 4;
  L.total = off;
  return L;
}

template <int C, int MAXT, int WPS>
__global__ __launch_bounds__(JAC_THREADS, WPS) void rc_jacobian_kernel(RcGeom g, int nb, int actk,
                                                                       const float* __restrict__ theta,
                                                                       const float* __restrict__ jf,
                                                                       const int8_t* __restrict__ s, int64_t ns,
                                                                       int64_t np, float* __restrict__ O,
                                                                       float* __restrict__ ws) {
  constexpr int CT = C / 16, CH = C / 4, P = 4 / CT, KEYSH = 8 / CH;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int N = g.N, NT = g.NT, npad = 16 * NT;
  const JacLds LY = jac_lds<C>(N);
  char* const buf0 = lds;
  char* const buf1 = lds + LY.bufb;
  uint16_t* const tabc = reinterpret_cast<uint16_t*>(lds + LY.tabc);
  uint16_t* const tabp = reinterpret_cast<uint16_t*>(lds + LY.tabp);
  float* const spf = reinterpret_cast<float*>(lds + LY.spf);
  float* const sred = reinterpret_cast<float*>(lds + LY.sred);
  const int tid = threadIdx.x, lane = tid % WAVE, wv = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int gq = lane / 16, l16 = lane % 16;
  const int m0 = wv % CT, part = wv / CT;  // weight gradient: output tile and position share of the wave
  const int64_t per = (int64_t)C * C * 9;
  // records of this workgroup: per block x and z1, [tile of the wave][ct][lane] of v4f
  const int64_t rec_arr = (int64_t)4 * MAXT * CT * WAVE;  // v4f entries of one array
  v4f* const rec = reinterpret_cast<v4f*>(ws) + (int64_t)blockIdx.x * 2 * nb * rec_arr + (int64_t)wv * MAXT * CT * WAVE;
  const float isq2 = 0.70710678118654752f;

  for (int e = tid; e < npad * 9; e += JAC_THREADS) {
    const int tap = e / npad, p = e - tap * npad;
    uint16_t v = 0;
    if (p < N) {
      const int src = tap_pos(g, p / g.L1, p % g.L1, tap);
      v = (uint16_t)(src * (C * 4) + (((src / KEYSH) & (CH - 1)) << 4));
    }
    tabc[tap * npad + p] = v;
    tabp[p * 16 + tap] = v;
  }

  auto site = [&](int k) { return 16 * (wv + 4 * k) + l16; };
  // wave-uniform; a wave has at least MAXT / 2 tiles (jac_maxt)
  auto has = [&](int k) { return k < MAXT / 2 || wv + 4 * k < NT; };
  int put_off[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
    put_off[ct] = l16 * (C * 4) + (((4 * ct + gq) ^ ((l16 / KEYSH) & (CH - 1))) << 4);
  auto put = [&](char* buf, int k, int ct, v4f v) {
    // the swizzle key of site 16 t + l16 depends on l16 alone
    if (site(k) < N) *reinterpret_cast<v4f*>(buf + (wv + 4 * k) * (16 * C * 4) + put_off[ct]) = v;
  };
  // acc[k][ct] += the 3 x 3 convolution of the positions in buf with layer l's fragments
  auto conv = [&](const char* buf, int l, int dir, v4f (&acc)[MAXT][CT]) {
    const v4f* fr = reinterpret_cast<const v4f*>(jf + ((int64_t)l * 2 + dir) * per) + lane;
    // an opaque zero: the 9 x MAXT table addresses are formed here, not
    // hoisted into registers held (or spilled) across the kernel
    int z0 = 0;
    asm volatile("" : "+v"(z0));
    const uint16_t* tc = tabc + z0 + site(0);
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
      v4f a[CT][CT];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int h = 0; h < CT; ++h) a[ct][h] = fr[((tap * CT + ct) * CT + h) * WAVE];
#pragma unroll
      for (int k = 0; k < MAXT; ++k) {
        if (MAXT == 1 || has(k)) {
          const uint32_t off = has(k) ? tc[tap * npad + 64 * k] : 0;
#pragma unroll
          for (int h = 0; h < CT; ++h) {
            const v4f b = *reinterpret_cast<const v4f*>(buf + (off ^ ((4 * h + gq) << 4)));
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
              for (int ct = 0; ct < CT; ++ct)
                acc[k][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[ct][h][j], b[j], acc[k][ct], 0, 0, 0);
          }
        }
      }
    }
    mfma_settle<MAXT * CT>(&acc[0][0]);
  };
  auto zero = [&](v4f (&acc)[MAXT][CT]) {
#pragma unroll
    for (int k = 0; k < MAXT; ++k)
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc[k][ct] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  };
  // offset of layer l's weights in theta (and in the O row); its bias follows
  auto w_off = [&](int l) { return l == 0 ? (int64_t)0 : (int64_t)10 * C + (l - 1) * (per + C); };
  auto bias4 = [&](int64_t b, int ct) { return *reinterpret_cast<const v4f*>(theta + b + 16 * ct + 4 * gq); };
  // sums over the positions of dz (registers, output layout) into sred[wv][c]
  auto bias_grad = [&](const v4f (&dz)[MAXT][CT]) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      v4f t = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < MAXT; ++k)
        if (has(k) && site(k) < N) t += dz[k][ct];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v = t[i];
        v = row_sum(v);
        if (l16 == 0) sred[wv * C + 16 * ct + 4 * gq + i] = v;
      }
    }
  };
  // weight gradient of a C -> C layer from dz (buf0) and its input (buf1) into
  // the O row; ends with the buffers free
  auto wgrad = [&](float* __restrict__ Ow, bool has_bias) {
    v4f acc[9][CT];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int h = 0; h < CT; ++h) acc[t][h] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const int cb = (l16 & 3) * 4;
    const uint32_t ca = (uint32_t)(4 * m0 + (l16 >> 2)) << 4;
    const int ksteps = (N + 3) / 4;
#pragma unroll 2
    for (int ks = part; ks < ksteps; ks += P) {
      const int p = 4 * ks + gq;  // < npad
      const v4i t0 = *reinterpret_cast<const v4i*>(tabp + p * 16);
      const int t8 = tabp[p * 16 + 8];
      const int o4 = (uint32_t)t0[2] & 0xffff;  // tap 4: the position itself
      float a = *reinterpret_cast<const float*>(buf0 + (o4 ^ ca) + cb);
      a = p < N ? a : 0.0f;
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const uint32_t off = t == 8 ? (uint32_t)t8 : ((t & 1) ? (uint32_t)t0[t / 2] >> 16 : (uint32_t)t0[t / 2] & 0xffff);
#pragma unroll
        for (int h = 0; h < CT; ++h) {
          const float b = *reinterpret_cast<const float*>(buf1 + (off ^ ((uint32_t)(4 * h + (l16 >> 2)) << 4)) + cb);
          acc[t][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc[t][h], 0, 0, 0);
        }
      }
    }
    __syncthreads();  // every wave has read both buffers
    // tap t of tile m0 is summed by part t % P; the other parts hand theirs over
    v4f* const slots = reinterpret_cast<v4f*>(lds);
    float* const out = reinterpret_cast<float*>(lds) + CT * 9 * CT * 256 * (P - 1);
#pragma unroll
    for (int t = 0; t < 9; ++t)
      if (t % P != part) {
        const int sl = part - (part > t % P ? 1 : 0);
#pragma unroll
        for (int h = 0; h < CT; ++h) slots[((((m0 * 9 + t) * CT + h) * (P - 1)) + sl) * WAVE + lane] = acc[t][h];
      }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 9; ++t)
      if (t % P == part) {
#pragma unroll
        for (int h = 0; h < CT; ++h) {
          v4f v = acc[t][h];
#pragma unroll
          for (int q = 0; q < P - 1; ++q) v += slots[((((m0 * 9 + t) * CT + h) * (P - 1)) + q) * WAVE + lane];
#pragma unroll
          for (int i = 0; i < 4; ++i) out[(16 * m0 + 4 * gq + i) * (C * 9) + (16 * h + l16) * 9 + t] = v[i];
        }
      }
    __syncthreads();
    for (int e = tid; e < C * C * 9; e += JAC_THREADS) Ow[e] = out[e];
    if (has_bias && tid < C) Ow[C * C * 9 + tid] = (sred[tid] + sred[C + tid]) + (sred[2 * C + tid] + sred[3 * C + tid]);
    __syncthreads();
  };

  for (int64_t n = blockIdx.x; n < ns; n += gridDim.x) {
    float* Orow = O + n * np;
    for (int p = tid; p < N; p += JAC_THREADS) spf[p] = (float)s[n * N + p];
    __syncthreads();
    v4f x[MAXT][CT];  // residual stream, then the running gradient
    // ---- forward with record
    for (int i = 0; i < nb; ++i) {
      const float sc = rsqrtf((float)(i + 1));
      const int64_t b1 = w_off(2 * i) + (i == 0 ? 9 * C : per), b2 = w_off(2 * i + 1) + per;
      v4f z[MAXT][CT];
      if (i == 0) {
#pragma unroll
        for (int k = 0; k < MAXT; ++k) {
          if (!has(k)) continue;
          int z0 = 0;
          asm volatile("" : "+v"(z0));
          const uint16_t* tc = tabc + z0 + site(k);
          float sv[9];
#pragma unroll
          for (int tap = 0; tap < 9; ++tap) sv[tap] = spf[tc[tap * npad] / (C * 4)] * isq2;
          const float spin = spf[site(k) < N ? site(k) : 0];
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            x[k][ct] = v4f{spin, spin, spin, spin};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const int co = 16 * ct + 4 * gq + q;
              float a = 0.0f;
#pragma unroll
              for (int tap = 0; tap < 9; ++tap) a += theta[co * 9 + tap] * sv[tap];
              z[k][ct][q] = a;
            }
          }
        }
      } else {
#pragma unroll
        for (int k = 0; k < MAXT; ++k) {
          if (!has(k)) continue;
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            rec[2 * i * rec_arr + (k * CT + ct) * WAVE + lane] = x[k][ct];
            put(buf0, k, ct, act4(x[k][ct], sc, actk));
          }
        }
        __syncthreads();
        zero(z);
        conv(buf0, 2 * i, 0, z);
      }
#pragma unroll
      for (int k = 0; k < MAXT; ++k) {
        if (!has(k)) continue;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const v4f v = z[k][ct] + bias4(b1, ct);
          rec[(2 * i + 1) * rec_arr + (k * CT + ct) * WAVE + lane] = v;
          put(buf1, k, ct, act4(v, 1.0f, actk));
        }
      }
      __syncthreads();
      zero(z);
      conv(buf1, 2 * i + 1, 0, z);
#pragma unroll
      for (int k = 0; k < MAXT; ++k)
        if (has(k))
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            if (i != nb - 1) z[k][ct] += bias4(b2, ct);
            x[k][ct] += z[k][ct];
          }
    }
    // ---- head: dX = softmax(h) / sqrt(nb + 1), h = x / sqrt(nb + 1)
    {
      const float hs = rsqrtf((float)(nb + 1));
      float m = -INFINITY;
#pragma unroll
      for (int k = 0; k < MAXT; ++k)
        if (has(k) && site(k) < N)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int q = 0; q < 4; ++q) m = fmaxf(m, x[k][ct][q] * hs);
      m = wave_max(m);
      if (lane == 0) sred[wv] = m;
      __syncthreads();
      m = fmaxf(fmaxf(sred[0], sred[1]), fmaxf(sred[2], sred[3]));
      float t = 0.0f;
#pragma unroll
      for (int k = 0; k < MAXT; ++k)
        if (has(k) && site(k) < N)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              x[k][ct][q] = expf(x[k][ct][q] * hs - m);
              t += x[k][ct][q];
            }
      t = wave_sum(t);
      if (lane == 0) sred[4 + wv] = t;
      __syncthreads();
      const float inv = 1.0f / (sred[4] + sred[5] + sred[6] + sred[7]) * hs;
#pragma unroll
      for (int k = 0; k < MAXT; ++k)
        if (has(k))
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) x[k][ct] *= inv;
      __syncthreads();  // sred and the buffers are free
    }
    // ---- backward
    for (int i = nb - 1; i >= 0; --i) {
      const float sc = rsqrtf((float)(i + 1));
      v4f d[MAXT][CT];
      // conv2: dz2 = dX, input a1 = act(z1)
#pragma unroll
      for (int k = 0; k < MAXT; ++k) {
        if (!has(k)) continue;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const v4f z1 = rec[(2 * i + 1) * rec_arr + (k * CT + ct) * WAVE + lane];
          put(buf1, k, ct, act4(z1, 1.0f, actk));
          put(buf0, k, ct, x[k][ct]);
        }
      }
      if (i != nb - 1) bias_grad(x);
      __syncthreads();
      zero(d);
      conv(buf0, 2 * i + 1, 1, d);
      wgrad(Orow + w_off(2 * i + 1), i != nb - 1);
      // dz1 = da1 act'(z1); conv1's input y = act(x_i sc)
#pragma unroll
      for (int k = 0; k < MAXT; ++k) {
        if (!has(k)) continue;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const v4f z1 = rec[(2 * i + 1) * rec_arr + (k * CT + ct) * WAVE + lane];
          d[k][ct] *= act_grad4(z1, 1.0f, actk);
          put(buf0, k, ct, d[k][ct]);
          if (i > 0) {
            const v4f xi = rec[2 * i * rec_arr + (k * CT + ct) * WAVE + lane];
            put(buf1, k, ct, act4(xi, sc, actk));
          }
        }
      }
      bias_grad(d);
      __syncthreads();
      if (i > 0) {
        zero(d);
        conv(buf0, 2 * i, 1, d);
        wgrad(Orow + w_off(2 * i), true);
#pragma unroll
        for (int k = 0; k < MAXT; ++k) {
          if (!has(k)) continue;
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            const v4f xi = rec[2 * i * rec_arr + (k * CT + ct) * WAVE + lane];
            x[k][ct] += d[k][ct] * act_grad4(xi, sc, actk) * sc;
          }
        }
      } else {
        // first layer (one input channel): G[co][tap], column lane%16 = tap
        v4f acc = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        const int tap = l16 < 9 ? l16 : 0;
        const int ksteps = (N + 3) / 4;
        for (int ks = part; ks < ksteps; ks += P) {
          const int p = 4 * ks + gq;
          const uint32_t o4 = tabp[p * 16 + 4];
          float a = *reinterpret_cast<const float*>(buf0 + (o4 ^ ((uint32_t)(4 * m0 + (l16 >> 2)) << 4)) + (l16 & 3) * 4);
          a = p < N ? a : 0.0f;
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, spf[tabp[p * 16 + tap] / (C * 4)] * isq2, acc, 0, 0, 0);
        }
        __syncthreads();
        v4f* const slots = reinterpret_cast<v4f*>(lds);
        slots[(m0 * P + part) * WAVE + lane] = acc;
        __syncthreads();
        for (int e = tid; e < C * 9; e += JAC_THREADS) {
          const int co = e / 9, t = e % 9, ln = ((co % 16) / 4) * 16 + t;
          float v = 0.0f;
          for (int q = 0; q < P; ++q) v += slots[((co / 16) * P + q) * WAVE + ln][co % 4];
          Orow[e] = v;
        }
        if (tid < C) Orow[9 * C + tid] = (sred[tid] + sred[C + tid]) + (sred[2 * C + tid] + sred[3 * C + tid]);
        __syncthreads();
      }
    }
  }
}

}  // namespace qtx

using namespace qtx;

// ================================================================ C ABI
extern "C" {

// tiles per wave of the Jacobian's kernel for this lattice
static int jac_maxt(const qtx_resconv_desc* d) {
  const int nt = (d->L0 * d->L1 + 15) / 16;
  return nt <= 4 ? 1 : (nt <= 8 ? 2 : (nt <= 16 ? 4 : 8));
}

// bytes of one workgroup's forward records
static size_t jac_slot_bytes(const qtx_resconv_desc* d) {
  return (size_t)2 * d->nblocks * 4 * jac_maxt(d) * (d->channels / 16) * WAVE * 16;
}

static int jac_launch(void* stream, const qtx_resconv_desc* d, const void* packed, const int8_t* s, int64_t ns,
                      float* O, void* ws, int64_t slots) {
  RcLayout L = rc_layout(d);
  RcGeom g{L.L0, L.L1, L.N, (L.N + 15) / 16, std::log((double)L.C * (double)L.N)};
  hipStream_t st = as_stream(stream);
  const float* theta = (const float*)packed;  // raw theta copy at offset 0
  const float* jf = (const float*)((const char*)packed + L.off_jac);
  const dim3 grid((unsigned)std::min<int64_t>(ns, slots));
  const int maxt = jac_maxt(d);
#define QTX_JAC(CC, MT, WPS)                                                                                       \
  do {                                                                                                             \
    const int lds = jac_lds<CC>(L.N).total;                                                                        \
    QTX_HIP(hipFuncSetAttribute((const void*)rc_jacobian_kernel<CC, MT, WPS>,                                      \
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds));                                 \
    hipLaunchKernelGGL((rc_jacobian_kernel<CC, MT, WPS>), grid, dim3(JAC_THREADS), lds, st, g, L.nb, L.actk, theta, \
                       jf, s, ns, L.nparams, O, (float*)ws);                                                       \
  } while (0)
  if (L.C == 16) {
    if (maxt == 1) QTX_JAC(16, 1, 3);
    else if (maxt == 2) QTX_JAC(16, 2, 3);
    else if (maxt == 4) QTX_JAC(16, 4, 3);
    else QTX_JAC(16, 8, 2);
  } else {
    if (maxt == 1) QTX_JAC(32, 1, 2);
    else if (maxt == 2) QTX_JAC(32, 2, 2);
    else if (maxt == 4) QTX_JAC(32, 4, 2);
    else QTX_JAC(32, 8, 1);
  }
#undef QTX_JAC
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

size_t qtx_resconv_jacobian_ws_bytes(const qtx_resconv_desc* d, int64_t ns) {
  if (rc_check(d) != QTX_OK || ns <= 0) return 0;
  return (size_t)std::min<int64_t>(ns, JAC_SLOTS) * jac_slot_bytes(d);
}

int qtx_resconv_jacobian(void* stream, const qtx_resconv_desc* d, const void* packed, const int8_t* s, int64_t ns,
                         float* O, void* ws, size_t ws_bytes) {
  int rc = rc_check(d);
  if (rc) return rc;
  QTX_REQUIRE(packed && ns >= 0 && (ns == 0 || (s && O)), "bad arguments");
  if (ns == 0) return QTX_OK;
  size_t need = qtx_resconv_jacobian_ws_bytes(d, ns);
  if (ws == nullptr || ws_bytes < need)
    return fail(QTX_EWORKSPACE, "workspace too small: need " + std::to_string(need) + " bytes");
  return jac_launch(stream, d, packed, s, ns, O, ws, JAC_SLOTS);
}

// ---------------------------------------------------------------- allocation-free Jacobian
// The per-sample forward records of qtx_resconv_jacobian_noalloc live in this
// file-scope device array (one copy per GPU, held until the process ends)
// instead of a caller workspace; a launch has as many workgroups as the array
// holds records for.  Host code uses the per-device address from
// hipGetSymbolAddress, never the array's name (a host-side stand-in).
constexpr size_t RC_JAC_SCRATCH_BYTES = (size_t)128 << 20;
static __device__ __align__(256) char scratch[RC_JAC_SCRATCH_BYTES];

namespace {
constexpr int RC_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[RC_MAX_DEVICES] = {};

// the calling thread's current device's copy of scratch
int jac_scratch(void** out) {
  int dev = 0;
  QTX_HIP(hipGetDevice(&dev));
  QTX_REQUIRE(dev >= 0 && dev < RC_MAX_DEVICES, "device index out of range");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    QTX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    QTX_REQUIRE(p != nullptr, "hipGetSymbolAddress returned no address for the Jacobian scratch");
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return QTX_OK;
}
}  // namespace

int qtx_resconv_jacobian_noalloc(void* stream, const qtx_resconv_desc* d, const void* packed, const int8_t* s,
                                 int64_t ns, float* O) {
  int rc = rc_check(d);
  if (rc) return rc;
  QTX_REQUIRE(packed && ns >= 0 && (ns == 0 || (s && O)), "bad arguments");
  void* ws = nullptr;
  rc = jac_scratch(&ws);
  if (rc) return rc;
  if (ns == 0) return QTX_OK;
  const size_t slot = jac_slot_bytes(d);
  if (slot > RC_JAC_SCRATCH_BYTES)
    return fail(QTX_EINVAL, "one sample's Jacobian records need " + std::to_string(slot) +
                                " bytes, more than the " + std::to_string(RC_JAC_SCRATCH_BYTES) +
                                "-byte scratch of the allocation-free entry point");
  return jac_launch(stream, d, packed, s, ns, O, ws, std::min<int64_t>(JAC_SLOTS, RC_JAC_SCRATCH_BYTES / slot));
}

}  // extern "C"
