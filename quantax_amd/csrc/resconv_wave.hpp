// ResConv forward on any lattice, with the Metropolis, E_loc and log psi
// kernels around it (the 16 x 16, 16-channel network and large 32-channel
// split-bf16 ones have kernels of their own in qtx_resconv.hip).
//
// P waves (1, 2 or 4) evaluate one configuration; a workgroup has 4 waves and
// 4 / P configurations.  A wave owns the 16-site tiles wq, wq + P, ... (at
// most MAXT) of its configuration and keeps their accumulators, residual
// stream and the LDS offsets of their taps' source sites in registers, so a
// layer reads its input from LDS, holds every output in registers and writes
// it back in place.  With P = 1 nothing is shared between waves: no barrier
// after the start of the kernel, every chain or candidate proceeds on its own
// and the waves of a SIMD overlap one's activations with another's MFMAs.
// P grows with the lattice (registers) and when there are too few
// configurations for the SIMDs (rw_pick).
//
// Per layer the K loop runs over the taps outside the tile loop: one tap's
// weights serve all tiles.  With 16 channels a layer's weights are in
// registers as a whole, and the next layer's are fetched while the activations
// run; with 32 they are fetched tap by tap.  The sums run in the order of the
// layout (bias, then tap, column half, K step), so a configuration's
// amplitude is the same bit for bit whichever P evaluates it; the head's
// log-sum-exp is merged tile by tile in four (eight on L0 x 16 lattices)
// interleaved classes for the same reason.
//
// Bound: MFMA issue and VALU (activation, split) in FP32; LDS reads of the
// activations (two 16-byte fragments per three MFMAs) in split-bf16 with 16
// channels.
// Measured against the previous any-lattice kernels (two configurations per
// workgroup, tap addresses formed per tile on VALU, ping-pong activations, a
// barrier per layer): J1-J2 E_loc of 1000 samples 10 x 10, 16 channels, 4
// blocks, FP32 16.4 -> 7.5 ms; a forward of 1000 6 x 6 configurations 50 -> 25
// us; forwards of 10000 6 x 6 configurations 533 -> 215 us, 8000 of 10 x 10 718 ->
// 360 us (split-bf16 323 -> 195), 3000 of 10 x 10 with 32 channels 554 -> 346 us
// (split-bf16 313 -> 142), 2000 of 18 x 18 510 -> 313 us.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "resconv.hpp"

namespace qtx {

constexpr int RW_THREADS = 256;

template <int C, int MODE>
struct RwK {
  static constexpr int CT = C / 16;
  static constexpr int CH = C / 4;                                       // 16-byte chunks per site
  static constexpr int KS = (MODE == QTX_CONV_BF16X3 && C == 16) ? 5 : 9;  // K steps = table rows used per site
  static constexpr int ROWS = (MODE == QTX_CONV_BF16X3 && C == 16) ? 10 : 9;  // rows of the source table
};

// byte offsets in a workgroup's dynamic LDS; G configurations
struct RwLds {
  int act, act_bytes;  // activations, per configuration
  int tab;             // [ROWS][npad] uint16: byte offset of the tap's source site, swizzle key in place
  int sp, sp_bytes;    // spins, per configuration
  int red;             // [G][NT + 8] float2
  int wq, tq;          // Metropolis: [G][64] proposal words (uint2), thresholds (double)
  int s0, vlist;       // E_loc: the sample, its valid candidates (int16)
  int total;
};

template <int C, int MODE>
__host__ __device__ inline RwLds rw_lds(int N, int G, int noff) {
  const int NT = (N + 15) / 16, npad = 16 * NT;
  RwLds L;
  int off = 0;
  L.act = off;
  L.act_bytes = npad * C * 4;
  off += G * L.act_bytes;
  L.tab = off;
  off += RwK<C, MODE>::ROWS * npad * 2;
  L.sp = off;
  L.sp_bytes = npad;
  off += G * npad;
  L.red = off;
  off += G * (NT + 8) * 8;
  L.wq = off;
  off += G * WAVE * 8;
  L.tq = off;
  off += G * WAVE * 8;
  L.s0 = off;
  off += npad;
  L.vlist = off;
  off += (noff * 2 + 15) / 16 * 16;
  L.total = off;
  return L;
}

template <int C, int MODE, int MAXT, int P, int MINT>
struct RwFwd {
  using K = RwK<C, MODE>;
  static constexpr int CT = K::CT, KS = K::KS;
  static constexpr bool BF = MODE == QTX_CONV_BF16X3;
  static constexpr bool WHOLE = C == 16;  // a layer's weights in registers
  static constexpr int NOFF = (MAXT * KS + 1) / 2;
  // the C = 32 split-bf16 head keeps a running (max, sum) per lane and class
  static constexpr bool LANE_HEAD = BF && C == 32;

  const RcArgs& a;
  int wq;          // wave of the configuration
  char* act;       // this configuration's activations
  const uint16_t* tab;
  const int8_t* sp;
  float2* red;     // [NT] tiles, then [8] classes
  uint32_t off[NOFF];  // source offsets of (K step, tile), two per register

  __device__ __forceinline__ bool has(int k) const { return k < MINT || wq + P * k < a.g.NT; }
  __device__ __forceinline__ static void sync() {
    if constexpr (P == 1) wave_lds_fence();
    else __syncthreads();
  }

  __device__ __forceinline__ void load_offsets() {
    const int lane = threadIdx.x % WAVE, npad = 16 * a.g.NT;
    auto at = [&](int e) -> uint32_t {
      const int ks = e / MAXT, k = e % MAXT;
      if (e >= MAXT * KS || !has(k)) return 0;
      const int row = (BF && C == 16) ? 2 * ks + (lane >> 5) : ks;
      return tab[row * npad + 16 * (wq + P * k) + lane % 16];
    };
#pragma unroll
    for (int i = 0; i < NOFF; ++i) off[i] = at(2 * i) | (at(2 * i + 1) << 16);
  }

  // log|psi| of the spins in sp (the same value in every lane of the
  // configuration's waves); par: the configuration's slot in a pair (sets the
  // merge classes), vw: number of classes.  With P > 1 every wave of the
  // workgroup calls it.
  __device__ __forceinline__ double run(int par, int vw) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // per-lane addresses formed inside the forward
    const int lane = tid % WAVE, gq = lane / 16, l16 = lane % 16;
    const int N = a.g.N, NT = a.g.NT, npad = 16 * NT, nb = a.nb, actk = a.actk;
    const float* pf = reinterpret_cast<const float*>(a.packed);
    constexpr int per = C * C * 9;
    constexpr int SHIFT = C == 16 ? 6 : 7;
    constexpr int KEY = 8 / K::CH;
    const int key = (l16 / KEY) & (K::CH - 1);
    auto valid = [&](int k) { return 16 * (wq + P * k) + l16 < N; };

    // ---- stores of four channels of a site
    int st[CT], st2[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      if constexpr (!BF) {
        st[ct] = l16 * (C * 4) + (((4 * ct + gq) ^ key) << 4);
        st2[ct] = 0;
      } else {
        st[ct] = l16 * (C * 4) + (((2 * ct + (gq >> 1)) ^ key) << 4) + (gq & 1) * 8;
        st2[ct] = l16 * (C * 4) + (((C / 8 + 2 * ct + (gq >> 1)) ^ key) << 4) + (gq & 1) * 8;
      }
    }
    auto put = [&](int k, int ct, v4f v) {
      char* base = act + (wq + P * k) * (16 * C * 4);
      if (valid(k)) {
        if constexpr (!BF) {
          *reinterpret_cast<v4f*>(base + st[ct]) = v;
        } else {
          v4bf hi, lo;
          split_bf16x4(v, hi, lo);
          *reinterpret_cast<v4bf*>(base + st[ct]) = hi;
          *reinterpret_cast<v4bf*>(base + st2[ct]) = lo;
        }
      }
    };

    // ---- weights and biases of a layer (C = 16: whole; C = 32: one tap)
    v4f wa[!BF ? (WHOLE ? KS : 1) * CT * CT : 1];
    v8bf wh[BF ? (WHOLE ? KS : 1) * CT : 1], wl[BF ? (WHOLE ? KS : 1) * CT : 1];
    v4f bias[CT];
    auto fetch = [&](int l, int ks, int slot) {
      if constexpr (!BF) {
        const v4f* fr = reinterpret_cast<const v4f*>(a.packed + a.off_jac) + (int64_t)l * 2 * per / 4 + lane;
#pragma unroll
        for (int e = 0; e < CT * CT; ++e) wa[slot * CT * CT + e] = fr[(ks * CT * CT + e) * WAVE];
      } else {
        const v8bf* fr = reinterpret_cast<const v8bf*>(a.packed + a.off_frag + (int64_t)l * a.frag_bytes) + 2 * lane;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          wh[slot * CT + ct] = fr[(ct * KS + ks) * 2 * WAVE];
          wl[slot * CT + ct] = fr[(ct * KS + ks) * 2 * WAVE + 1];
        }
      }
    };
    auto fetch_layer = [&](int l) {
      if constexpr (WHOLE) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) fetch(l, ks, ks);
      } else {
        fetch(l, 0, 0);
      }
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        bias[ct] = *reinterpret_cast<const v4f*>(pf + a.bias_off + (int64_t)l * C + 16 * ct + 4 * gq);
    };
    fetch_layer(1);

    // ---- layer 0: one input channel, s / sqrt(2), on VALU
    v4f res[MAXT][CT];
    {
      const float* W0 = pf + a.off_l0w + 4 * gq * 9;
      const float* b0 = pf + a.off_l0b + 4 * gq;
      int z0 = 0;
      asm volatile("" : "+v"(z0));  // table addresses are formed per forward
      const uint16_t* tz = tab + z0 + 16 * wq + l16;
#pragma unroll
      for (int k = 0; k < MAXT; ++k) {
        if (has(k)) {
          float sv[9];
#pragma unroll
          for (int tap = 0; tap < 9; ++tap)
            sv[tap] = (float)sp[tz[tap * npad + 16 * P * k] >> SHIFT] * 0.70710678118654752f;
          const float spin = (float)sp[valid(k) ? 16 * (wq + P * k) + l16 : 0];
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            v4f z;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              float v = b0[16 * ct + q];
#pragma unroll
              for (int tap = 0; tap < 9; ++tap) v += W0[(16 * ct + q) * 9 + tap] * sv[tap];
              z[q] = v;
            }
            res[k][ct] = v4f{spin, spin, spin, spin};
            put(k, ct, act4(z, 1.0f, actk));
          }
        }
      }
    }
    sync();

    // ---- layers 1 .. 2 nb - 1
    for (int l = 1; l < 2 * nb; ++l) {
      const bool is_conv2 = (l % 2) == 1, last = l == 2 * nb - 1;
      v4f acc[MAXT][CT];
#pragma unroll
      for (int k = 0; k < MAXT; ++k)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[k][ct] = bias[ct];
      // unpacked per layer, not hoisted out of the layer loop
#pragma unroll
      for (int i = 0; i < NOFF; ++i) asm volatile("" : "+v"(off[i]));
      // The MFMAs, unrolled for the wave's tile count: no branch inside, since
      // the compiler counts the wait states behind an MFMA along the
      // fall-through path only
      auto mfmas = [&](auto count) {
        constexpr int n = decltype(count)::value;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int slot = WHOLE ? ks : 0;
          v4f ca[!BF ? CT * CT : 1];
          v8bf ch[BF ? CT : 1], cl[BF ? CT : 1];
          if constexpr (!BF) {
#pragma unroll
            for (int e = 0; e < CT * CT; ++e) ca[e] = wa[slot * CT * CT + e];
          } else {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
              ch[ct] = wh[slot * CT + ct];
              cl[ct] = wl[slot * CT + ct];
            }
          }
          if constexpr (!WHOLE)
            if (ks + 1 < KS) fetch(l, ks + 1, 0);
#pragma unroll
          for (int k = 0; k < n; ++k) {
            const int e = ks * MAXT + k;
            const uint32_t o = (e & 1) ? off[e / 2] >> 16 : off[e / 2] & 0xffff;
            if constexpr (!BF) {
#pragma unroll
              for (int h = 0; h < CT; ++h) {
                const v4f b = *reinterpret_cast<const v4f*>(act + (o ^ ((4 * h + gq) << 4)));
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                  for (int ct = 0; ct < CT; ++ct)
                    acc[k][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(ca[ct * CT + h][j], b[j], acc[k][ct], 0, 0, 0);
              }
            } else {
              const int jh = C == 16 ? (gq & 1) : gq;
              const v8bf bh = *reinterpret_cast<const v8bf*>(act + (o ^ (jh << 4)));
              const v8bf bl = *reinterpret_cast<const v8bf*>(act + (o ^ ((C / 8 + jh) << 4)));
#pragma unroll
              for (int ct = 0; ct < CT; ++ct) {
                acc[k][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cl[ct], bh, acc[k][ct], 0, 0, 0);
                acc[k][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ch[ct], bl, acc[k][ct], 0, 0, 0);
                acc[k][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ch[ct], bh, acc[k][ct], 0, 0, 0);
              }
            }
          }
        }
        mfma_settle<n * CT>(&acc[0][0]);
      };
      const int mine = (NT - wq + P - 1) / P;  // tiles of this wave
      if (mine == MAXT) mfmas(std::integral_constant<int, MAXT>{});
      if constexpr (MAXT - 1 >= (MINT > 1 ? MINT : 1))
        if (mine == MAXT - 1) mfmas(std::integral_constant<int, MAXT - 1>{});
      if constexpr (MAXT - 2 >= (MINT > 1 ? MINT : 1))
        if (mine == MAXT - 2) mfmas(std::integral_constant<int, MAXT - 2>{});
      if constexpr (MAXT - 3 >= (MINT > 1 ? MINT : 1))
        if (mine == MAXT - 3) mfmas(std::integral_constant<int, MAXT - 3>{});
      if constexpr (MAXT - 4 >= (MINT > 1 ? MINT : 1))
        if (mine == MAXT - 4) mfmas(std::integral_constant<int, MAXT - 4>{});
      if (!last) {
        fetch_layer(l + 1);
        if constexpr (P > 1) __syncthreads();  // every wave has read this layer's input
        else wave_lds_fence();
        const float scale = is_conv2 ? rsqrtf((float)(l / 2 + 2)) : 1.0f;
#pragma unroll
        for (int k = 0; k < MAXT; ++k) {
          if (has(k)) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
              v4f x = acc[k][ct];
              if (is_conv2) {
                x += res[k][ct];
                res[k][ct] = x;
              }
              put(k, ct, act4(x, scale, actk));
            }
          }
        }
        sync();
        continue;
      }
      // ---- head: h = (z + r) / sqrt(nb + 1), log-sum-exp over channels and sites
      const float scale = rsqrtf((float)(nb + 1));
      if constexpr (LANE_HEAD) {
        constexpr int NC = 4 / P;  // classes of this wave: tiles t = wq + P c mod 4
        float m_l[NC], s_l[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          m_l[c] = -INFINITY;
          s_l[c] = 0.0f;
        }
#pragma unroll
        for (int k = 0; k < MAXT; ++k) {
          if (has(k) && valid(k)) {
            const int c = k % NC;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
              float hv[4];
#pragma unroll
              for (int q = 0; q < 4; ++q) hv[q] = (acc[k][ct][q] + res[k][ct][q]) * scale;
              const float mn = fmaxf(m_l[c], fmaxf(fmaxf(hv[0], hv[1]), fmaxf(hv[2], hv[3])));
              float sacc = s_l[c] * __expf(m_l[c] - mn);
#pragma unroll
              for (int q = 0; q < 4; ++q) sacc += __expf(hv[q] - mn);
              s_l[c] = sacc;
              m_l[c] = mn;
            }
          }
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const float m_w = wave_max(m_l[c]);
          const float s_w = wave_sum(m_l[c] > -INFINITY ? s_l[c] * __expf(m_l[c] - m_w) : 0.0f);
          if (lane == 0) red[NT + wq + P * c] = make_float2(m_w, s_w);
        }
        sync();
      } else {
#pragma unroll
        for (int k = 0; k < MAXT; ++k) {
          if (has(k)) {
            float m = -INFINITY, hv[CT * 4];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const float h = (acc[k][ct][q] + res[k][ct][q]) * scale;
                hv[ct * 4 + q] = h;
                if (valid(k)) m = fmaxf(m, h);
              }
            m = wave_max(m);
            float sacc = 0.0f;
            if (valid(k)) {
#pragma unroll
              for (int i = 0; i < CT * 4; ++i) sacc += __expf(hv[i] - m);
            }
            sacc = wave_sum(sacc);
            if (lane == 0) red[wq + P * k] = make_float2(m, sacc);
          }
        }
        sync();
        if (wq == 0 && lane < vw) {
          float m_b = -INFINITY, s_b = 0.0f;
          for (int t = (lane - par * NT) & (vw - 1); t < NT; t += vw) {
            const float m = red[t].x, sacc = red[t].y;
            const float mm = fmaxf(m_b, m);
            s_b = s_b * __expf(m_b - mm) + sacc * __expf(m - mm);
            m_b = mm;
          }
          red[NT + lane] = make_float2(m_b, s_b);
        }
        sync();
      }
    }
    // the classes' (max, sum) merged in FP32, the same in every lane
    const int nc = LANE_HEAD ? 4 : vw;
    float m = -INFINITY;
    for (int w = 0; w < nc; ++w) m = fmaxf(m, red[NT + w].x);
    float ssum = 0.0f;
    for (int w = 0; w < nc; ++w) {
      const float mw = red[NT + w].x;
      if (mw > -INFINITY) ssum += red[NT + w].y * __expf(mw - m);
    }
    return (double)m + (double)logf(ssum) - a.g.log_cn;
  }
};

// The source table: by every thread of the workgroup, barrier after it.  A site per
// thread and one division for its nine taps: a workgroup forms it for 4 / P forwards
// (1300 of 10 x 16, one block, FP32: 31.1 -> 28.3 us against a division per entry)
template <int C, int MODE>
__device__ __forceinline__ void rw_build_tab(const RcGeom& g, uint16_t* tab) {
  using K = RwK<C, MODE>;
  const int npad = 16 * g.NT;
  for (int p = threadIdx.x; p < npad; p += RW_THREADS) {
    const int y = p / g.L1, x = p - y * g.L1;
    const int ym = y == 0 ? g.L0 - 1 : y - 1, yp = y + 1 == g.L0 ? 0 : y + 1;
    const int xm = x == 0 ? g.L1 - 1 : x - 1, xp = x + 1 == g.L1 ? 0 : x + 1;
#pragma unroll
    for (int row = 0; row < K::ROWS; ++row) {
      const int ys = row / 3 == 0 ? ym : (row / 3 == 1 ? y : yp), xs = row % 3 == 0 ? xm : (row % 3 == 1 ? x : xp);
      const int src = row < 9 ? ys * g.L1 + xs : p;  // row 9: zero weights, any finite input
      const int v = src * (C * 4) + (((src / (8 / K::CH)) & (K::CH - 1)) << 4);
      tab[row * npad + p] = (uint16_t)(p < g.N ? v : 0);
    }
  }
}

// merge classes of the head and whether configurations pair up in them
struct RwMerge {
  int vw, pair;
};

template <int C, int MODE, int MAXT, int P, int MINT>
__global__ __launch_bounds__(RW_THREADS, 2) void rw_logpsi_kernel(RcArgs a, RwMerge mg, const int8_t* __restrict__ s,
                                                                  int64_t ns, double* __restrict__ logabs) {
  constexpr int G = 4 / P;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const RwLds L = rw_lds<C, MODE>(a.g.N, G, 0);
  const int lane = threadIdx.x % WAVE, wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int grp = wv / P, N = a.g.N;
  uint16_t* tab = reinterpret_cast<uint16_t*>(lds + L.tab);
  rw_build_tab<C, MODE>(a.g, tab);
  const int64_t c0 = xcd_block(blockIdx.x, gridDim.x) * G;
  for (int i = threadIdx.x; i < G * N; i += RW_THREADS) {
    const int b = i / N, j = i - b * N;
    lds[L.sp + b * L.sp_bytes + j] = (c0 + b < ns) ? s[(c0 + b) * N + j] : (int8_t)1;
  }
  __syncthreads();
  const int64_t c = c0 + grp;
  if (P == 1 && c >= ns) return;
  RwFwd<C, MODE, MAXT, P, MINT> f{a, wv % P, lds + L.act + grp * L.act_bytes, tab,
                                  reinterpret_cast<const int8_t*>(lds + L.sp + grp * L.sp_bytes),
                                  reinterpret_cast<float2*>(lds + L.red) + grp * (a.g.NT + 8), {}};
  f.load_offsets();
  const double lp = f.run((int)(c & 1) & mg.pair, mg.vw);
  if (wv % P == 0 && lane == 0 && c < ns) logabs[c] = lp;
}

// Metropolis: as rc_metropolis_kernel (null proposals run no forward, words 64
// steps at a time); the flips of a proposal are applied to the chain's spins
// and taken back on rejection.
template <int C, int MODE, int MAXT, int P, int MINT>
__global__ __launch_bounds__(RW_THREADS, 2) void rw_metropolis_kernel(
    RcArgs a, RwMerge mg, int kind, const int32_t* __restrict__ nbr, int width, int hopping,
    const uint32_t* __restrict__ words, int nsteps, int64_t ns, double reweight, double tie_tol,
    int8_t* __restrict__ s, double* __restrict__ logabs, int32_t* __restrict__ n_accept,
    int32_t* __restrict__ n_near) {
  constexpr int G = 4 / P;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ int mv_upd[G];
  const RwLds L = rw_lds<C, MODE>(a.g.N, G, 0);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), grp = wv / P, wq = wv % P;
  const int N = a.g.N;
  uint16_t* tab = reinterpret_cast<uint16_t*>(lds + L.tab);
  rw_build_tab<C, MODE>(a.g, tab);
  const int64_t c0 = xcd_block(blockIdx.x, gridDim.x) * G;  // per-chain Philox words of a step share lines
  for (int i = threadIdx.x; i < G * N; i += RW_THREADS) {
    const int b = i / N, j = i - b * N;
    lds[L.sp + b * L.sp_bytes + j] = (c0 + b < ns) ? s[(c0 + b) * N + j] : (int8_t)1;
  }
  __syncthreads();
  const int64_t c = c0 + grp;
  if (P == 1 && c >= ns) return;
  int8_t* cur = reinterpret_cast<int8_t*>(lds + L.sp + grp * L.sp_bytes);
  uint2* wq_s = reinterpret_cast<uint2*>(lds + L.wq) + grp * WAVE;
  double* tq_s = reinterpret_cast<double*>(lds + L.tq) + grp * WAVE;
  RwFwd<C, MODE, MAXT, P, MINT> f{a, wq, lds + L.act + grp * L.act_bytes, tab, cur,
                                  reinterpret_cast<float2*>(lds + L.red) + grp * (a.g.NT + 8), {}};
  f.load_offsets();
  double lp_cur = (c < ns) ? logabs[c] : 0.0;
  int n_hop = 0, acc_n = 0, near_n = 0, tc = 0;
  {
    const int lane = threadIdx.x % WAVE;
    int cnt = 0;
    for (int i = lane; i < N; i += WAVE) cnt += (cur[i] == hopping);
    n_hop = wave_sum(cnt);
  }
  for (;;) {
    int lane = threadIdx.x % WAVE;
    asm volatile("" : "+v"(lane));
    int fa = -1, fb = -1;
    bool upd = false;
    double thr = 0.0;
    if (wq == 0) {
      while (c < ns && tc < nsteps && !upd) {
        const int q = tc % WAVE;
        if (q == 0) {
          if (tc + lane < nsteps) {
            const uint4 w = reinterpret_cast<const uint4*>(words)[(int64_t)(tc + lane) * ns + c];
            wq_s[lane] = make_uint2(w.x, w.y);
            tq_s[lane] = accept_threshold(w.z, w.w);
          }
          wave_lds_fence();
        }
        const uint2 w = wq_s[q];
        propose_move(kind, cur, N, nbr, width, hopping, n_hop, w.x, w.y, lane, fa, fb, upd);
        thr = tq_s[q];
        ++tc;
      }
      if (upd && lane == 0) {
        cur[fa] = -cur[fa];
        if (fb >= 0) cur[fb] = -cur[fb];
      }
    }
    if constexpr (P == 1) {
      if (!upd) break;
      wave_lds_fence();
    } else {
      if (wq == 0 && lane == 0) mv_upd[grp] = upd ? 1 : 0;
      __syncthreads();
      int any = 0;
#pragma unroll
      for (int b = 0; b < G; ++b) any |= mv_upd[b];
      if (!any) break;
    }
    const double lp_new = f.run((int)(c & 1) & mg.pair, mg.vw);
    if (wq == 0 && upd) {
      const double d = reweight * (lp_new - lp_cur);
      const bool acc = (d > thr) || (lp_cur == -INFINITY);
      near_n += fabs(d - thr) < tie_tol ? 1 : 0;
      if (acc) {
        lp_cur = lp_new;
        acc_n += 1;
      } else if (lane == 0) {
        cur[fa] = -cur[fa];
        if (fb >= 0) cur[fb] = -cur[fb];
      }
      wave_lds_fence();
    }
  }
  const int lane = threadIdx.x % WAVE;
  if (c < ns && wq == 0) {
    for (int i = lane; i < N; i += WAVE) s[c * N + i] = cur[i];
    if (lane == 0) {
      logabs[c] = lp_cur;
      n_accept[c] += acc_n;
      n_near[c] += near_n;
    }
  }
}

// E_loc: workgroup (sample n, run sp of S) as in rc_eloc_kernel; configuration
// slot grp takes candidates first + grp, first + grp + G, ... of the run.
template <int C, int MODE, int MAXT, int P, int MINT>
__global__ __launch_bounds__(RW_THREADS, 2) void rw_eloc_kernel(RcArgs a, RwMerge mg, qtx_ham H,
                                                                const int8_t* __restrict__ s,
                                                                const double* __restrict__ logabs, int S,
                                                                double* __restrict__ eloc,
                                                                int32_t* __restrict__ nconn) {
  constexpr int G = 4 / P;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ int nvalid_s;
  __shared__ double diag_s, e_s[G];
  const RwLds L = rw_lds<C, MODE>(a.g.N, G, H.noff);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), grp = wv / P, wq = wv % P;
  const int N = a.g.N;
  const int64_t n = blockIdx.x / (unsigned)S;
  const int sp = (int)(blockIdx.x % (unsigned)S);
  uint16_t* tab = reinterpret_cast<uint16_t*>(lds + L.tab);
  int8_t* s0 = reinterpret_cast<int8_t*>(lds + L.s0);
  int16_t* vlist = reinterpret_cast<int16_t*>(lds + L.vlist);
  rw_build_tab<C, MODE>(a.g, tab);
  for (int i = threadIdx.x; i < N; i += RW_THREADS) {
    const int8_t v = s[n * N + i];
    s0[i] = v;
    for (int b = 0; b < G; ++b) lds[L.sp + b * L.sp_bytes + i] = v;
  }
  __syncthreads();
  if (wv == 0) {
    // diagonal part and the ordered list of valid candidates (ballot compaction)
    const int lane = threadIdx.x;
    const double dg = diag_energy(H, s0, lane);
    int pos = 0;
    for (int base = 0; base < H.noff; base += WAVE) {
      const int k = base + lane;
      const bool v = (k < H.noff) && cand_valid(H, s0, k);
      const uint64_t m = __ballot(v);
      const uint64_t below = (lane == 0) ? 0ull : (m & ((~0ull) >> (64 - lane)));
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
  const int nbatch = (nall + G - 1) / G;
  const int first = (int)((int64_t)nbatch * sp / S) * G;
  const int stop = (int)((int64_t)nbatch * (sp + 1) / S) * G;
  const int end = stop < nall ? stop : nall;
  const double lp0 = logabs[n];
  int8_t* cfg = reinterpret_cast<int8_t*>(lds + L.sp + grp * L.sp_bytes);
  RwFwd<C, MODE, MAXT, P, MINT> f{a, wq, lds + L.act + grp * L.act_bytes, tab, cfg,
                                  reinterpret_cast<float2*>(lds + L.red) + grp * (a.g.NT + 8), {}};
  f.load_offsets();
  double e = 0.0;
  // the candidate's sites and coupling are fetched one forward ahead
  int na = -1, nb = -1;
  double nc = 0.0;
  auto next = [&](int j) {
    na = nb = -1;
    nc = 0.0;
    if (j < end) {
      const int k = vlist[j];
      na = H.off_a[k];
      nb = H.off_b[k];
      nc = H.off_c[k];
    }
  };
  next(first + grp);
  // P = 1: every wave counts its own candidates; P > 1: the workgroup's waves
  // take the same number of turns
  for (int j = first + grp; (P == 1 ? j : j - grp) < end; j += G) {
    int lane = threadIdx.x % WAVE;
    asm volatile("" : "+v"(lane));
    const int fa = na, fb = nb;
    const double cf = nc;
    if (wq == 0 && lane == 0) {
      if (fa >= 0) cfg[fa] = -s0[fa];
      if (fb >= 0) cfg[fb] = -s0[fb];
    }
    next(j + G);
    f.sync();
    const double lp = f.run((j & 1) & mg.pair, mg.vw);
    if (fa >= 0) e += cf * exp_ratio(lp - lp0);
    if (wq == 0 && lane == 0) {
      if (fa >= 0) cfg[fa] = s0[fa];
      if (fb >= 0) cfg[fb] = s0[fb];
    }
    if constexpr (P == 1) wave_lds_fence();
  }
  if (threadIdx.x % WAVE == 0 && wq == 0) e_s[grp] = e;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
#pragma unroll
    for (int b = 0; b < G; ++b) t += e_s[b];
    eloc[blockIdx.x] = (sp == 0) ? diag_s + t : t;
    if (nconn && sp == 0) nconn[n] = nall;
  }
}

// ---------------------------------------------------------------- dispatch
// Waves per configuration and tiles per wave.  P = 1 (2 where the tiles'
// registers would not leave two waves per SIMD) does the least work, but a pass
// then takes as long as one wave needs for a whole network, for 1 to 1024
// configurations (one wave per SIMD) and half as long again up to 2048; P = 4
// takes time in proportion, in steps of 256 (a workgroup per CU).  So P = 4 is
// for fewer than 768 and between 1025 and 1536.  us, P = 4 | P = 1, four blocks:
//                       768         1000        1250        1640        2000
//   6 x 6, 16, FP32   22 | 25     31 | 25     35 | 37     48 | 37     53 | 37
//   8 x 8, 16, FP32   24 | 31     32 | 31     37 | 47     51 | 47     56 | 47
//   8 x 8, 32, bf16   31 | 42     51 | 41     57 | 50     76 | 50     83 | 52
//   10 x 10, 16, FP32 37 | 49     51 | 49     60 | 78     83 | 78     92 | 78
//   12 x 12, 16 (P 2) 55 | 56     66 | 57     85 | 89    116 | 110   131 | 112
// (10 x 10 in split-bf16 at 1000: 31 | 34, so five to eight tiles start at 1537.)
// A single tile leaves three of four waves idle: P = 1 from 512 on.  In a sweep the
// chains whose proposal does not move leave their waves' time to the others, so
// P = 4 stays best up to 1536 (8 x 8, FP32, 24 steps of 1000 chains: 535 | 625 us;
// of 2000: 949 | 855) and P = 2 starts at 1793.
// A forward of 16 channels in FP32 (fp32 set) goes by its tiles too: P = 4 leaves half the
// waves of two tiles idle, half those of the second turn with five and six, the last
// turn's with nine and more, where 768 and 1280 configurations (three and five per CU)
// do not hide it.  us, one | four | eight blocks, P = 4 and the choice here: 2 x 16 at 1300
// 12.6 | 34.7 | 62.7 and 9.1 | 27.4 | 51.3; 6 x 16 at 1000 14.8 | 46.0 | 88.3 and 12.8 | 42.6
// | 81.9; 10 x 16 at 1300 28.2 | 103.5 | 204 and 24.0 | 91.1 | 181; 14 x 14 32.2 | 125 | 246
// and 29.7 | 117 | 234.  Split-bf16 loses up to a tenth by it.
struct RwPick {
  int P, maxt;
};
inline RwPick rw_pick(int C, int N, int64_t units, bool sweep = false, bool fp32 = false) {
  const int nt = (N + 15) / 16;
  if (fp32 && C == 16) {
    if (nt == 2 && units > 768) return {1, 4};
    if (nt > 4 && nt <= 6 && units > 768 && units <= 1024) return {1, 8};
    if (nt > 8 && nt <= 16 && units > 1280) return {2, 8};
  }
  const bool late = units > 1536, full = late || (!sweep && units > 768 && units <= 1024);
  if (nt == 1 && units >= 512) return {1, 4};
  if (full && nt <= 4) return {1, 4};
  if (C == 16) {
    if (late && nt <= 8) return {1, 8};
    if ((sweep ? units > 1792 : full) && nt > 8 && nt <= 16) return {2, 8};
    return {4, nt <= 8 ? 2 : (nt <= 16 ? 4 : 8)};
  }
  if (units > 1792 && nt <= 8) return {2, 4};
  return {4, nt <= 8 ? 2 : (nt <= 16 ? 4 : 7)};
}

// The choice for a local energy of ns samples: about a quarter of an exchange
// Hamiltonian's candidates are valid.  On one or two tiles, where P = 4 leaves two or
// three waves of each configuration idle, a table too short to be split over workgroups
// with P = 4 (eloc_split) takes P = 1, four candidates at a time (us, 16 channels, four
// blocks, P = 4 | P = 1, 3 to 200 samples: transverse-field Ising 3 x 5 FP32 140 | 45,
// split-bf16 112 | 35, 4 x 8 309 | 135, 250 | 94; Heisenberg 3 x 5 168 | 55, 134 | 42; split
// in two or more, 4 x 8 104 | 167, 85 | 116).
inline RwPick rw_eloc_pick(int C, int N, int64_t noff, int64_t ns) {
  if (C == 16 && N <= 32 && noff < 64) return {1, 4};
  return rw_pick(C, N, ns * (noff / 4));
}

inline RwMerge rw_merge(const RcLayout& L) {
  return RwMerge{(L.C == 16 && L.L1 == 16 && L.L0 <= 16) ? 8 : 4, (L.C == 16 && L.N <= 256) ? 1 : 0};
}

template <int C, int MODE>
int rw_logpsi(hipStream_t st, const RcLayout& L, const RcArgs& a, const int8_t* s, int64_t ns, double* logabs);
template <int C, int MODE>
int rw_metropolis(hipStream_t st, const RcLayout& L, const RcArgs& a, int kind, const int32_t* nbr, int width,
                  int hopping, const uint32_t* words, int nsteps, int64_t ns, double reweight, double tie_tol,
                  int8_t* s, double* logabs, int32_t* n_accept, int32_t* n_near);
template <int C, int MODE>
int rw_eloc(hipStream_t st, const RcLayout& L, const RcArgs& a, const qtx_ham& H, const int8_t* s,
            const double* logabs, int64_t ns, int S, double* eloc, int32_t* nconn);

// the instance of FN for L's channels and precision
#define RW_CALL(FN, L, ...)                                                                        \
  ((L).C == 16 ? ((L).mode == QTX_CONV_FP32 ? FN<16, QTX_CONV_FP32>(__VA_ARGS__)                   \
                                            : FN<16, QTX_CONV_BF16X3>(__VA_ARGS__))                \
               : ((L).mode == QTX_CONV_FP32 ? FN<32, QTX_CONV_FP32>(__VA_ARGS__)                   \
                                            : FN<32, QTX_CONV_BF16X3>(__VA_ARGS__)))

// KERNEL<C, MODE, MAXT, P, MINT> on a grid of GRID (G = 4 / P configurations
// per workgroup in scope); MINT: tiles every wave has, from the class's least
// tile count
#define RW_LAUNCH(KERNEL, C, MODE, MAXT, P, MINT, NOFF, GRID, ...)                                              \
  do {                                                                                                          \
    constexpr int G = 4 / P;                                                                                    \
    const int lds_ = rw_lds<C, MODE>(L.N, G, NOFF).total;                                                       \
    QTX_HIP(hipFuncSetAttribute((const void*)KERNEL<C, MODE, MAXT, P, MINT>,                                    \
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds_));                             \
    hipLaunchKernelGGL((KERNEL<C, MODE, MAXT, P, MINT>), dim3((unsigned)(GRID)), dim3(RW_THREADS), lds_, st, a, \
                       rw_merge(L), __VA_ARGS__);                                                               \
  } while (0)

}  // namespace qtx
