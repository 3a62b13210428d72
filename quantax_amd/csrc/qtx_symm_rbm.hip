// Symmetry-projected RBM_Dense in float64 without materialised images:
// psi_sym(s) = sum_g c_g prod_i cosh((W T_g s + b)_i) (symmetry/symmetry.py:343-392
// over model/shallow_nets.py:35-126), and a whole Metropolis sweep of it in one
// launch (sampler/metropolis.py:246-322).
//
// One workgroup (1 to 8 waves) per configuration.  u = W T_g s for 16
// permutations at a time is an FP64-MFMA product: W stays in registers as A
// fragments for the whole launch (M <= 64, N <= 64), the B operand is the
// spins gathered from LDS through the permutation table, and an image and its
// spin inversion share u (h = b +- u).  A lane then holds up to 16 hidden
// units of one permutation: it sums |h| and multiplies the factors
// (1 + e^(-2|h|)) / 2 in [1/2, 1], so an image takes one logarithm instead of
// one per unit.
//
// Bound: FP64 VALU (the exponentials, about 40 instructions each).  72 steps
// of 256 chains plus E_loc, 6 x 6, M = 36, 576 images: 25.4 -> 1.5 ms against
// images -> forward -> projection as separate launches, which also evaluated
// the proposals that leave the spins unchanged.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "common.hpp"

namespace qtx {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int SR_MAXW = 8;            // waves of a workgroup
constexpr int SR_TAB_BYTES = 49152;   // permutation table in LDS

struct SymRbmArgs {
  const double* packed;  // [Wt (N, M) | b (M)]
  int M, N;
  const int32_t* perm;   // (nperm, N)
  int nperm, z2;
  const double* coef;    // nperm (2 nperm with z2)
};

template <int MT, int KS>
struct SymRbm {
  const SymRbmArgs& a;
  uint8_t* tab;    // [tile][KS][64]: source site of (permutation, site) as the B fragment wants it
  double* spd;     // 4 KS spins as +-1.0 (0 past N)
  double* la;      // [tile][2][16] log-amplitudes of the images
  double* red;     // 2 x SR_MAXW
  double wf[MT][KS], bf[MT][4];
  int nt, nw;

  __device__ __forceinline__ void init() {
    const int lane = threadIdx.x % WAVE;
    nt = (a.nperm + 15) / 16;
    nw = blockDim.x / WAVE;
    for (int e = threadIdx.x; e < nt * KS * WAVE; e += blockDim.x) {
      const int l = e % WAVE, ks = (e / WAVE) % KS, t = e / WAVE / KS;
      const int p = 16 * t + l % 16, j = 4 * ks + l / 16;
      tab[e] = (p < a.nperm && j < a.N) ? (uint8_t)a.perm[(int64_t)p * a.N + j] : (uint8_t)(j < a.N ? j : 4 * KS - 1);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int i = 16 * mt + lane % 16;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int j = 4 * ks + lane / 16;
        wf[mt][ks] = (i < a.M && j < a.N) ? a.packed[(int64_t)j * a.M + i] : 0.0;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = 16 * mt + 4 * q + lane / 16;
        bf[mt][q] = r < a.M ? a.packed[(int64_t)a.M * a.N + r] : 0.0;
      }
    }
  }

  // log-amplitudes of the images +-T_p s of this lane's permutation, summed
  // over the four lane groups that share it
  __device__ __forceinline__ void image(const v4d (&u)[MT], double s, double& l) {
    double sum = 0.0, prod = 1.0;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (16 * mt + 4 * q < a.M) {  // rows past M have h = 0: factor 1, nothing to add
          const double h = fabs(fma(s, u[mt][q], bf[mt][q]));
          sum += h;
          prod *= fma(0.5, exp(-2.0 * h), 0.5);
        }
    sum += __shfl_xor(sum, 16, WAVE);
    prod *= __shfl_xor(prod, 16, WAVE);
    sum += __shfl_xor(sum, 32, WAVE);
    prod *= __shfl_xor(prod, 32, WAVE);
    l = sum + log(prod);
  }

  // sign and log|psi_sym| of the spins in spd, in every thread; every thread
  // of the workgroup calls it, with a barrier between the spins' writes and it
  __device__ __forceinline__ void eval(double& sg, double& lo) {
    const int lane = threadIdx.x % WAVE, wv = threadIdx.x / WAVE;
    double m = -INFINITY;
    for (int t = wv; t < nt; t += nw) {
      v4d u[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) u[mt] = v4d{0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const double b = spd[tab[(t * KS + ks) * WAVE + lane]];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) u[mt] = __builtin_amdgcn_mfma_f64_16x16x4f64(wf[mt][ks], b, u[mt], 0, 0, 0);
      }
      // wait out the last MFMA before the branches of image(): the compiler
      // counts its wait states along the fall-through path only
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+v"(u[mt]));
      asm volatile("s_nop 15\n\ts_nop 15" : "+v"(u[0]));
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+v"(u[mt]));
      double lp, lm = -INFINITY;
      image(u, 1.0, lp);
      if (a.z2) image(u, -1.0, lm);
      const int p = 16 * t + lane % 16;
      if (lane < 32) {  // group 0: the permutation, group 1: its inversion
        const bool inv = lane >= 16;
        const double l = inv ? lm : lp;
        const bool ok = p < a.nperm && (!inv || a.z2);
        la[t * 32 + lane] = l;
        if (ok && a.coef[inv ? a.nperm + p : p] != 0.0) m = fmax(m, l);
      }
    }
    m = wave_max(m);
    if (lane == 0) red[wv] = m;
    __syncthreads();
    m = red[0];
    for (int w = 1; w < nw; ++w) m = fmax(m, red[w]);
    double acc = 0.0;
    if (m > -INFINITY) {
      for (int t = wv; t < nt; t += nw) {
        const int p = 16 * t + lane % 16;
        const bool inv = lane >= 16;
        if (lane < 32 && p < a.nperm && (!inv || a.z2))
          acc += a.coef[inv ? a.nperm + p : p] * exp(la[t * 32 + lane] - m);
      }
    }
    acc = wave_sum(acc);
    if (lane == 0) red[SR_MAXW + wv] = acc;
    __syncthreads();
    double S = 0.0;
    for (int w = 0; w < nw; ++w) S += red[SR_MAXW + w];
    sg = (S > 0.0) ? 1.0 : (S < 0.0 ? -1.0 : 0.0);
    lo = (S != 0.0) ? m + log(fabs(S)) : -INFINITY;
  }
};

struct SymRbmLds {
  int tab, spd, la, red, total;
};
template <int KS>
__host__ __device__ inline SymRbmLds sym_rbm_lds(int nperm) {
  const int nt = (nperm + 15) / 16;
  SymRbmLds L;
  int off = 0;
  L.tab = off;
  off += nt * KS * WAVE;
  L.spd = off;
  off += 4 * KS * 8 + 8;
  L.la = off;
  off += nt * 32 * 8;
  L.red = off;
  off += 2 * SR_MAXW * 8;
  L.total = off;
  return L;
}

template <int MT, int KS>
__global__ __launch_bounds__(SR_MAXW * 64, 2) void sym_rbm_logpsi_kernel(SymRbmArgs a, const int8_t* __restrict__ s,
                                                                         int64_t ns, double* __restrict__ sign,
                                                                         double* __restrict__ logabs) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const SymRbmLds L = sym_rbm_lds<KS>(a.nperm);
  SymRbm<MT, KS> f{a, reinterpret_cast<uint8_t*>(lds + L.tab), reinterpret_cast<double*>(lds + L.spd),
                   reinterpret_cast<double*>(lds + L.la), reinterpret_cast<double*>(lds + L.red)};
  f.init();
  for (int64_t n = blockIdx.x; n < ns; n += gridDim.x) {
    if (threadIdx.x < 4 * KS) f.spd[threadIdx.x] = (int)threadIdx.x < a.N ? (double)s[n * a.N + threadIdx.x] : 0.0;
    __syncthreads();
    double sg, lo;
    f.eval(sg, lo);
    if (threadIdx.x == 0) {
      sign[n] = sg;
      logabs[n] = lo;
    }
  }
}

// One workgroup per chain; the flips of a proposal are applied to the spins
// and taken back on rejection; a proposal that leaves them unchanged is never
// accepted and not evaluated.
template <int MT, int KS>
__global__ __launch_bounds__(SR_MAXW * 64, 2) void sym_rbm_metropolis_kernel(
    SymRbmArgs a, int kind, const int32_t* __restrict__ nbr, int width, int hopping,
    const uint32_t* __restrict__ words, int nsteps, int64_t ns, double reweight, double tie_tol,
    int8_t* __restrict__ s, double* __restrict__ sign, double* __restrict__ logabs, int32_t* __restrict__ n_accept,
    int32_t* __restrict__ n_near) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ int8_t cur[4 * KS];
  __shared__ uint2 wq[WAVE];
  __shared__ double tq[WAVE];
  __shared__ int mv[3];
  __shared__ double mv_thr;
  const SymRbmLds L = sym_rbm_lds<KS>(a.nperm);
  SymRbm<MT, KS> f{a, reinterpret_cast<uint8_t*>(lds + L.tab), reinterpret_cast<double*>(lds + L.spd),
                   reinterpret_cast<double*>(lds + L.la), reinterpret_cast<double*>(lds + L.red)};
  f.init();
  const int64_t c = xcd_block(blockIdx.x, gridDim.x);  // per-chain Philox words of a step share lines
  const int lane = threadIdx.x % WAVE, wv = threadIdx.x / WAVE, N = a.N;
  if (threadIdx.x < 4 * KS) {
    const int8_t v = (int)threadIdx.x < N ? s[c * N + threadIdx.x] : (int8_t)0;
    cur[threadIdx.x] = v;
    f.spd[threadIdx.x] = (double)v;
  }
  __syncthreads();
  int n_hop = 0;
  if (kind == QTX_EXCHANGE) {
    int cnt = 0;
    for (int i = lane; i < N; i += WAVE) cnt += (cur[i] == hopping);
    n_hop = wave_sum(cnt);
  }
  double lp = logabs[c], sg = sign[c];
  int acc_n = 0, near_n = 0, tc = 0;
  for (;;) {
    if (wv == 0) {
      int fa = -1, fb = -1;
      bool upd = false;
      double thr = 0.0;
      while (tc < nsteps && !upd) {
        const int q = tc % WAVE;
        if (q == 0) {
          if (tc + lane < nsteps) {
            const uint4 w = reinterpret_cast<const uint4*>(words)[(int64_t)(tc + lane) * ns + c];
            wq[lane] = make_uint2(w.x, w.y);
            tq[lane] = log1p(-words_to_uniform(w.z, w.w));
          }
          wave_lds_fence();
        }
        const uint2 w = wq[q];
        propose_move(kind, cur, N, nbr, width, hopping, n_hop, w.x, w.y, lane, fa, fb, upd);
        thr = tq[q];
        ++tc;
      }
      if (lane == 0) {
        mv[0] = fa;
        mv[1] = fb;
        mv[2] = upd ? 1 : 0;
        mv_thr = thr;
        if (upd) {
          f.spd[fa] = -f.spd[fa];
          if (fb >= 0) f.spd[fb] = -f.spd[fb];
        }
      }
    }
    __syncthreads();
    const int fa = mv[0], fb = mv[1];
    const double thr = mv_thr;
    if (!mv[2]) break;
    double sgn, ln;
    f.eval(sgn, ln);
    const double d = reweight * (ln - lp);
    const bool acc = (d > thr) || (lp == -INFINITY);
    near_n += fabs(d - thr) < tie_tol ? 1 : 0;
    if (acc) {
      lp = ln;
      sg = sgn;
      acc_n += 1;
    }
    if (threadIdx.x == 0) {
      if (acc) {
        cur[fa] = -cur[fa];
        if (fb >= 0) cur[fb] = -cur[fb];
      } else {
        f.spd[fa] = -f.spd[fa];
        if (fb >= 0) f.spd[fb] = -f.spd[fb];
      }
    }
    if (wv == 0) wave_lds_fence();
  }
  if ((int)threadIdx.x < N) s[c * N + threadIdx.x] = cur[threadIdx.x];
  if (threadIdx.x == 0) {
    logabs[c] = lp;
    sign[c] = sg;
    n_accept[c] += acc_n;
    n_near[c] += near_n;
  }
}

}  // namespace qtx

using namespace qtx;

static int ks_class(int N) { return N <= 16 ? 4 : (N <= 36 ? 9 : 16); }

// W's fragments fit in registers (M, N <= 64) and the permutation table in LDS
static bool sym_rbm_ok(int M, int N, int nperm) {
  return M >= 1 && M <= 64 && N >= 1 && N <= 64 && nperm >= 1 &&
         (int64_t)((nperm + 15) / 16) * ks_class(N) * WAVE <= SR_TAB_BYTES;
}

static int sym_rbm_check(const SymRbmArgs& a) {
  QTX_REQUIRE(a.packed && a.perm && a.coef, "null pointer");
  QTX_REQUIRE(sym_rbm_ok(a.M, a.N, a.nperm), "shape not supported (M, N <= 64, at most 768 tiles of the table)");
  return QTX_OK;
}

// KERNEL<MT, KS> with one workgroup per configuration of min(8, tiles) waves
#define SYM_LAUNCH(KERNEL, MT, KS, GRID, ...)                                                                       \
  do {                                                                                                              \
    const int lds_ = sym_rbm_lds<KS>(a.nperm).total;                                                                \
    QTX_HIP(hipFuncSetAttribute((const void*)KERNEL<MT, KS>, hipFuncAttributeMaxDynamicSharedMemorySize, lds_));    \
    hipLaunchKernelGGL((KERNEL<MT, KS>), dim3((unsigned)(GRID)), dim3(64 * std::min(SR_MAXW, (a.nperm + 15) / 16)), \
                       lds_, st, a, __VA_ARGS__);                                                                   \
  } while (0)
#define SYM_KS(KERNEL, MT, GRID, ...)                                          \
  do {                                                                         \
    if (ks == 4) SYM_LAUNCH(KERNEL, MT, 4, GRID, __VA_ARGS__);                 \
    else if (ks == 9) SYM_LAUNCH(KERNEL, MT, 9, GRID, __VA_ARGS__);            \
    else SYM_LAUNCH(KERNEL, MT, 16, GRID, __VA_ARGS__);                        \
  } while (0)
#define SYM_DISPATCH(KERNEL, GRID, ...)                                        \
  do {                                                                         \
    const int ks = ks_class(a.N);                                              \
    if (a.M <= 16) SYM_KS(KERNEL, 1, GRID, __VA_ARGS__);                       \
    else if (a.M <= 32) SYM_KS(KERNEL, 2, GRID, __VA_ARGS__);                  \
    else if (a.M <= 48) SYM_KS(KERNEL, 3, GRID, __VA_ARGS__);                  \
    else SYM_KS(KERNEL, 4, GRID, __VA_ARGS__);                                 \
  } while (0)

extern "C" {

int qtx_symm_rbm_supported(int32_t M, int32_t N, int32_t nperm) { return sym_rbm_ok(M, N, nperm) ? 1 : 0; }

int qtx_symm_rbm_logpsi(void* stream, const double* packed, int32_t M, int32_t N, const int32_t* perm, int32_t nperm,
                        int32_t z2, const double* coef, const int8_t* s, int64_t ns, double* sign, double* logabs) {
  const SymRbmArgs a{packed, M, N, perm, nperm, z2 ? 1 : 0, coef};
  int rc = sym_rbm_check(a);
  if (rc) return rc;
  QTX_REQUIRE(ns >= 0 && (ns == 0 || (s && sign && logabs)), "bad arguments");
  if (ns == 0) return QTX_OK;
  hipStream_t st = as_stream(stream);
  // persistent: the table and the fragments are set up once per workgroup
  SYM_DISPATCH(sym_rbm_logpsi_kernel, std::min<int64_t>(ns, 1024), s, ns, sign, logabs);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

int qtx_symm_rbm_metropolis(void* stream, const double* packed, int32_t M, int32_t N, const int32_t* perm,
                            int32_t nperm, int32_t z2, const double* coef, int kind, const int32_t* nbr, int32_t width,
                            int32_t hopping, const uint32_t* words, int32_t nsteps, int64_t ns, double reweight,
                            double tie_tol, int8_t* s, double* sign, double* logabs, int32_t* n_accept,
                            int32_t* n_near) {
  const SymRbmArgs a{packed, M, N, perm, nperm, z2 ? 1 : 0, coef};
  int rc = sym_rbm_check(a);
  if (rc) return rc;
  QTX_REQUIRE(kind == QTX_LOCALFLIP || kind == QTX_EXCHANGE, "kind must be QTX_LOCALFLIP or QTX_EXCHANGE");
  QTX_REQUIRE(kind == QTX_LOCALFLIP || (nbr != nullptr && width > 0), "EXCHANGE needs a neighbour table");
  QTX_REQUIRE(hopping == 1 || hopping == -1, "hopping must be +1 or -1");
  QTX_REQUIRE(nsteps >= 0 && ns >= 0 && ns <= 0x7fffffff, "bad size");
  QTX_REQUIRE(ns == 0 || (s && sign && logabs && n_accept && n_near && (nsteps == 0 || words)), "null pointer");
  if (ns == 0) return QTX_OK;
  hipStream_t st = as_stream(stream);
  SYM_DISPATCH(sym_rbm_metropolis_kernel, ns, kind, nbr, width, hopping, words, nsteps, ns, reweight, tie_tol, s, sign,
               logabs, n_accept, n_near);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

}  // extern "C"
