// RBM_Dense device bodies shared by the single-job kernels (qtx_core.hip) and
// the grouped serving kernels (qtx_serve.hip), so a chain evolves through the
// same instructions whichever launch carries it.
//
// packed = [Wt (N, M) | b (M)]: the column W[:, j] touched by a flip of site j
// is one contiguous row of Wt.  One wavefront owns one chain / sample; lane l
// holds hidden units l, l + 64, ... (R = ceil(M / 64) registers per lane).
#pragma once
#include <type_traits>

#include "common.hpp"

namespace qtx {

constexpr int MAXN = 1024;
constexpr int WAVES_PER_BLOCK = 4;

// copy one sample's spins into LDS (wave-cooperative)
__device__ __forceinline__ void load_spins(int8_t* sl, const int8_t* src, int N, int lane) {
  for (int i = lane; i < N; i += WAVE) sl[i] = src[i];
}

// h for lane-owned hidden units: h[r] = b[i] + sum_j Wt[j, i] s_j,  i = lane + 64 r
template <typename T, int R>
__device__ __forceinline__ void rbm_hidden(const T* __restrict__ Wt, const T* __restrict__ b, int M, int N,
                                           const int8_t* sl, int lane, T (&h)[R]) {
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int i = lane + WAVE * r;
    h[r] = (i < M) ? b[i] : T(0);
  }
  // J rows in flight at once, added in order: one row at a time, the wave waits
  // for the L2 in every one (4096 samples, 100 x 400: 90 -> 36 us).  Lanes past M load
  // nothing, because a load takes the L1 for as many lanes as it has (8192 samples, us
  // with the last unit's weights in their place | without: 36 x 144 FP64 41 | 33, 100 x
  // 400 188 | 163, FP32 63 | 54).  Single rows, whose many loads a branch on the lane
  // each would hold up (1000 samples, 100 x 1000 FP64: 62 | 77), branch on registers
  // that lie past M as a whole, where there are two of them at least (100 x 513, 1000
  // and 32768 samples: 57, 1404 | 53, 850; x 800 58, 1415 | 68, 1191; x 960 60, 1417 |
  // 76, 1357)
  constexpr int J = sizeof(T) * R <= 16 ? 8 : sizeof(T) * R <= 32 ? 4 : sizeof(T) * R <= 64 ? 2 : 1;
  int j = 0;
  auto batches = [&](auto skip) {
    for (; j + J <= N; j += J) {
      T w[J][R];
      const T* row = Wt + (int64_t)j * M + lane;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (skip.value && (J > 1 ? lane : 0) + WAVE * r >= M) continue;
#pragma unroll
        for (int u = 0; u < J; ++u) w[u][r] = row[u * M + (lane + WAVE * r < M ? WAVE * r : M - 1 - lane)];
      }
#pragma unroll
      for (int u = 0; u < J; ++u) {
        const T sj = (T)sl[j + u];
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (lane + WAVE * r < M) h[r] += w[u][r] * sj;
      }
      __builtin_amdgcn_sched_barrier(0);  // no second batch in registers
    }
  };
  if (J == 1 && M > WAVE * (R - 2)) batches(std::false_type{});
  else batches(std::true_type{});
  for (; j < N; ++j) {
    T sj = (T)sl[j];
    const T* row = Wt + (int64_t)j * M;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      int i = lane + WAVE * r;
      if (i < M) h[r] += row[i] * sj;
    }
  }
}

template <typename T, int R>
__device__ __forceinline__ double rbm_sum_logcosh(const T (&h)[R], int M, int lane) {
  T acc = T(0);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int i = lane + WAVE * r;
    if (i < M) acc += logcosh(h[r]);
  }
  return wave_sum((double)acc);
}

// log|psi| of one sample (and optionally its h row)
template <typename T, int R>
__device__ __forceinline__ void rbm_chain_logpsi(const T* __restrict__ packed, int M, int N, const int8_t* src,
                                                 int8_t* sl, int lane, double* logabs, T* h_out) {
  load_spins(sl, src, N, lane);
  __builtin_amdgcn_wave_barrier();
  const T* Wt = packed;
  const T* b = packed + (int64_t)M * N;
  T h[R];
  rbm_hidden<T, R>(Wt, b, M, N, sl, lane, h);
  double la = rbm_sum_logcosh<T, R>(h, M, lane);
  if (lane == 0) *logabs = la;
  if (h_out) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      int i = lane + WAVE * r;
      if (i < M) h_out[i] = h[r];
    }
  }
}

// the rows of Wt that a move of sites fa and fb (-1: none) needs, lane-owned
// hidden units (lanes past M: the last one's), all loads in flight at once
template <typename T, int R>
__device__ __forceinline__ void rbm_load_rows(const T* __restrict__ Wt, int M, int fa, int fb, int lane, T (&a)[R],
                                              T (&b)[R]) {
  const T* ra = Wt + (int64_t)fa * M;
  const T* rb = Wt + (int64_t)(fb >= 0 ? fb : fa) * M;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = lane + WAVE * r < M ? lane + WAVE * r : M - 1;
    a[r] = ra[i];
    b[r] = rb[i];
  }
}

// whether the rows of the next move are fetched during this one's log cosh: where
// the two rows' registers leave four waves per SIMD
template <typename T, int R>
constexpr bool rbm_rows_ahead() {
  return sizeof(T) == 4 ? R <= 8 : R <= 2;
}

// nsteps Metropolis steps of one chain with h resident in registers.
// getw(t) -> uint4 Philox block of step t.  s is read and written back;
// *logabs receives the local-update value; counters are incremented.
//
// VALU-bound (log cosh of the hidden units of every proposal that moves).  64
// steps are prepared at once, lane l step t0 + l: its words, its acceptance
// threshold (one FP64 log1p for 64 steps) and its move on the current spins
// (pos: the sites that hold `hopping`, in order).  A ballot then gives the next
// step that changes the spins; the moves are looked up again after an accepted
// exchange.  4096 chains x 200 exchanges, 400 hidden units: 872 -> 638 us.
template <typename T, int R, typename GetW>
__device__ __forceinline__ void rbm_chain_metropolis(const T* __restrict__ packed, int M, int N, int kind,
                                                     const int32_t* __restrict__ nbr, int width, int hopping,
                                                     int nsteps, GetW getw, double reweight, double tie_tol,
                                                     int8_t* s, int8_t* sl, uint16_t* pos, int lane, double* logabs,
                                                     int32_t* n_accept, int32_t* n_near) {
  load_spins(sl, s, N, lane);
  __builtin_amdgcn_wave_barrier();
  const T* Wt = packed;
  const T* b = packed + (int64_t)M * N;
  T h[R];
  rbm_hidden<T, R>(Wt, b, M, N, sl, lane, h);
  double lp = rbm_sum_logcosh<T, R>(h, M, lane);
  const bool ex = kind == QTX_EXCHANGE;
  int acc_count = 0, near_count = 0;
  constexpr bool AHEAD = rbm_rows_ahead<T, R>();
  T ra[R], rb[R];
  for (int t0 = 0; t0 < nsteps; t0 += WAVE) {
    const int cnt = nsteps - t0 < WAVE ? nsteps - t0 : WAVE;
    uint4 w = make_uint4(0, 0, 0, 0);
    if (lane < cnt) w = getw(t0 + lane);
    const double thr_l = accept_threshold(w.z, w.w);
    uint64_t todo = ~0ull >> (WAVE - cnt), moves = 0;
    int site = 0, nb = -1;
    int ca = -1, cb = -1;  // the move whose rows ra, rb hold
    bool look = true;
    while (todo != 0) {
      if (look) {
        bool moved;
        if (ex) {
          moved = false;
          const int n_hop = list_sites(sl, N, hopping, pos, lane);
          if (n_hop > 0) {
            site = pos[bounded(w.x, (uint32_t)n_hop)];
            nb = nbr[site * width + (int)bounded(w.y, (uint32_t)width)];
            moved = nb >= 0 && nb != site && sl[nb] != hopping;  // s' == s is never accepted (metropolis.py:314-316)
          }
        } else {
          site = (int)bounded(w.x, (uint32_t)N);
          moved = true;
        }
        moves = __ballot(moved);
        look = false;
      }
      const uint64_t left = moves & todo;
      if (left == 0) break;
      const int i = __ffsll((unsigned long long)left) - 1;
      todo &= ~((2ull << i) - 1);
      const int fa = __builtin_amdgcn_readlane(site, i), fb = ex ? __builtin_amdgcn_readlane(nb, i) : -1;
      const T sa = ex ? (T)hopping : (T)sl[fa];
      const T sb = ex ? (T)sl[fb] : T(0);
      if (!AHEAD || fa != ca || fb != cb) rbm_load_rows<T, R>(Wt, M, fa, fb, lane, ra, rb);
      T hn[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        int i = lane + WAVE * r;
        T v = h[r];
        if (i < M) {
          v -= T(2) * ra[r] * sa;
          if (fb >= 0) v -= T(2) * rb[r] * sb;
        }
        hn[r] = v;
      }
      // the rows of the step after a rejection, on their way during the log cosh
      const uint64_t next = moves & todo;
      ca = cb = -1;
      if (AHEAD && next != 0) {
        const int i = __ffsll((unsigned long long)next) - 1;
        ca = __builtin_amdgcn_readlane(site, i);
        cb = ex ? __builtin_amdgcn_readlane(nb, i) : -1;
        rbm_load_rows<T, R>(Wt, M, ca, cb, lane, ra, rb);
      }
      double lpn = rbm_sum_logcosh<T, R>(hn, M, lane);
      const double thr = readlane_f64(thr_l, i);
      double d = reweight * (lpn - lp);
      bool accept = (d > thr) || (lp == -INFINITY);
      near_count += (fabs(d - thr) < tie_tol) ? 1 : 0;
      if (accept) {
        acc_count += 1;
#pragma unroll
        for (int r = 0; r < R; ++r) h[r] = hn[r];
        lp = lpn;
        wave_lds_fence();
        if (lane == 0) {
          sl[fa] = -sl[fa];
          if (fb >= 0) sl[fb] = -sl[fb];
        }
        wave_lds_fence();
        look = ex;
      }
    }
  }
  __builtin_amdgcn_wave_barrier();
  for (int i = lane; i < N; i += WAVE) s[i] = sl[i];
  if (lane == 0) {
    *logabs = lp;
    *n_accept += acc_count;
    *n_near += near_count;
  }
}

// E_loc of one sample with local updates of h over the valid candidates: 64
// candidates are looked at at once, lane l candidate k0 + l, and the exponentials
// of the ones that connect are taken together at the end of the 64 (one FP64
// exp instead of one per candidate).  4096 samples, 400 hidden units, 200
// bonds: 934 -> 692 us.
template <typename T, int R>
__device__ __forceinline__ void rbm_sample_eloc(const T* __restrict__ packed, int M, int N, const qtx_ham& H,
                                                const int8_t* src, int8_t* sl, int lane, double* eloc,
                                                int32_t* nconn) {
  load_spins(sl, src, N, lane);
  __builtin_amdgcn_wave_barrier();
  const T* Wt = packed;
  const T* b = packed + (int64_t)M * N;
  T h[R], lc0[R];
  rbm_hidden<T, R>(Wt, b, M, N, sl, lane, h);
#pragma unroll
  for (int r = 0; r < R; ++r) lc0[r] = (lane + WAVE * r < M) ? logcosh(h[r]) : T(0);
  const double diag = diag_energy(H, sl, lane);
  double e = 0.0;
  int cnt = 0;
  for (int k0 = 0; k0 < H.noff; k0 += WAVE) {
    const int k = k0 + lane;
    const bool valid = k < H.noff && cand_valid(H, sl, k);
    const int la = valid ? H.off_a[k] : 0, lb = valid ? H.off_b[k] : -1;
    uint64_t left = __ballot(valid);
    cnt += __popcll(left);
    double dlp_l = 0.0;
    T ra[R], rb[R];
    int fa = 0, fb = -1;
    auto fetch = [&]() {  // the rows of the first candidate left
      const int i = __ffsll((unsigned long long)left) - 1;
      fa = __builtin_amdgcn_readlane(la, i);
      fb = __builtin_amdgcn_readlane(lb, i);
      rbm_load_rows<T, R>(Wt, M, fa, fb, lane, ra, rb);
    };
    constexpr bool AHEAD = rbm_rows_ahead<T, R>();
    if (AHEAD && left != 0) fetch();
    while (left != 0) {
      if (!AHEAD) fetch();
      const int i = __ffsll((unsigned long long)left) - 1;
      left &= left - 1;
      T sa = (T)sl[fa];
      T sb = (fb >= 0) ? (T)sl[fb] : T(0);
      T v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        v[r] = h[r] - T(2) * ra[r] * sa;
        if (fb >= 0) v[r] -= T(2) * rb[r] * sb;
      }
      if (AHEAD && left != 0) fetch();  // on their way during the log cosh
      T dl = T(0);
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (lane + WAVE * r < M) dl += logcosh(v[r]) - lc0[r];
      const double dlp = wave_sum((double)dl);
      dlp_l = lane == i ? dlp : dlp_l;
    }
    if (valid) e += H.off_c[k] * exp(dlp_l);
  }
  e = diag + wave_sum(e);
  if (lane == 0) {
    *eloc = e;
    if (nconn) *nconn = cnt;
  }
}

// one O row [tanh(h) (x) s, tanh(h)] by a whole block: tanh(h) into LDS, then a
// coalesced write of the row.  tl / tld / sl: block-shared scratch of MAXN.
template <typename T, typename TO>
__device__ __forceinline__ void rbm_jacobian_row(const T* __restrict__ packed, int M, int N, const int8_t* src,
                                                 TO* __restrict__ row, float* tl, double* tld, int8_t* sl) {
  const T* Wt = packed;
  const T* b = packed + (int64_t)M * N;
  for (int j = threadIdx.x; j < N; j += blockDim.x) sl[j] = src[j];
  __syncthreads();
  for (int i = threadIdx.x; i < M; i += blockDim.x) {
    T h = b[i];
    for (int j = 0; j < N; ++j) h += Wt[(int64_t)j * M + i] * (T)sl[j];
    T t = tanh(h);
    tl[i] = (float)t;
    tld[i] = (double)t;
  }
  __syncthreads();
  int64_t np = (int64_t)M * N + M;
  for (int64_t k = threadIdx.x; k < np; k += blockDim.x) {
    TO v;
    if (k < (int64_t)M * N) {
      int i = (int)(k / N), j = (int)(k % N);
      if (sizeof(TO) == 8)
        v = (TO)(tld[i] * (double)sl[j]);
      else
        v = (TO)(tl[i] * (float)sl[j]);
    } else {
      int i = (int)(k - (int64_t)M * N);
      v = (sizeof(TO) == 8) ? (TO)tld[i] : (TO)tl[i];
    }
    row[k] = v;
  }
  __syncthreads();  // the scratch is reused by the block's next row
}

}  // namespace qtx
