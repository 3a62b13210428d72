// Shared device helpers and error plumbing for libqtxhip (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string>

#include "../../include/qtx_hip.h"

namespace qtx {

void set_error(const std::string& msg);
int fail(int code, const std::string& msg);
int hip_check(hipError_t e, const char* what);

#define QTX_REQUIRE(cond, msg)                         \
  do {                                                 \
    if (!(cond)) return ::qtx::fail(QTX_EINVAL, msg); \
  } while (0)

#define QTX_HIP(call)                                   \
  do {                                                  \
    int _rc = ::qtx::hip_check((call), #call);          \
    if (_rc != QTX_OK) return _rc;                      \
  } while (0)

#define QTX_LAUNCH_CHECK() QTX_HIP(hipGetLastError())

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

constexpr int WAVE = 64;

// ---------------------------------------------------------------- reductions
// The xor-butterfly over lane distances 32, 16, 8, 4, 2, 1.  32-bit values go
// without the LDS crossbar: the two halves, then the odd and even rows of 16
// lanes, are exchanged by v_permlane{32,16}_swap, the rest by DPP row
// rotations (after the exchange at distance 2d a row is periodic in 2d lanes,
// so rotating by d reads lane ^ d).  Every lane of the wave must be active.
// The operands of each step are those of the __shfl_xor form, so sums are the
// same bit for bit (10 x 10 FP32 E_loc, which reduces in the head of every
// forward: 17.0 -> 16.4 ms).  64-bit values keep the crossbar: their kernels
// are bound by VALU issue, where two moves a step cost more than the LDS
// round trip they save (10 x 10 RBM sweep +2 %, 6 x 6 symmetric sweep +1 %).
template <int STEP>
__device__ __forceinline__ uint32_t lane_xor32(uint32_t v) {  // STEP 8, 4, 2, 1
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x120 + STEP, 0xf, 0xf, true);
}

template <typename T, typename F>
__device__ __forceinline__ T wave_butterfly(T v, F op) {
  if constexpr (sizeof(T) == 4) {
    uint32_t u = __builtin_bit_cast(uint32_t, v);
    auto h = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    u = __builtin_bit_cast(uint32_t, op(__builtin_bit_cast(T, (uint32_t)h[0]), __builtin_bit_cast(T, (uint32_t)h[1])));
    h = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    v = op(__builtin_bit_cast(T, (uint32_t)h[0]), __builtin_bit_cast(T, (uint32_t)h[1]));
    v = op(v, __builtin_bit_cast(T, lane_xor32<8>(__builtin_bit_cast(uint32_t, v))));
    v = op(v, __builtin_bit_cast(T, lane_xor32<4>(__builtin_bit_cast(uint32_t, v))));
    v = op(v, __builtin_bit_cast(T, lane_xor32<2>(__builtin_bit_cast(uint32_t, v))));
    v = op(v, __builtin_bit_cast(T, lane_xor32<1>(__builtin_bit_cast(uint32_t, v))));
  } else {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = op(v, __shfl_xor(v, off, WAVE));
  }
  return v;
}

// sum over each row of 16 lanes
__device__ __forceinline__ float row_sum(float v) {
  v += __builtin_bit_cast(float, lane_xor32<8>(__builtin_bit_cast(uint32_t, v)));
  v += __builtin_bit_cast(float, lane_xor32<4>(__builtin_bit_cast(uint32_t, v)));
  v += __builtin_bit_cast(float, lane_xor32<2>(__builtin_bit_cast(uint32_t, v)));
  v += __builtin_bit_cast(float, lane_xor32<1>(__builtin_bit_cast(uint32_t, v)));
  return v;
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  return wave_butterfly(v, [](T a, T b) { return a + b; });
}

// wave_sum(a * b) with the first step fused, a b + (a b of lane ^ 32): what the
// product form of the butterfly rounds to under FP contraction
__device__ __forceinline__ float wave_sum_prod(float a, float b) {
  const uint32_t u = __builtin_bit_cast(uint32_t, a * b);
  const auto h = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const uint32_t other = (threadIdx.x % WAVE) < 32 ? (uint32_t)h[1] : (uint32_t)h[0];
  uint32_t v = __builtin_bit_cast(uint32_t, fmaf(a, b, __builtin_bit_cast(float, other)));
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return row_sum(__builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]));
}

template <typename T>
__device__ __forceinline__ T wave_max(T v) {
  return wave_butterfly(v, [](T a, T b) { return (T)fmax(a, b); });
}

// Orders this wave's LDS writes before its later LDS reads (other lanes' data)
// for the compiler; the hardware runs a wave's LDS instructions in order.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ double readlane_f64(double v, int l) {
  const int2 u = __builtin_bit_cast(int2, v);
  const int2 s = int2{__builtin_amdgcn_readlane(u.x, l), __builtin_amdgcn_readlane(u.y, l)};
  return __builtin_bit_cast(double, s);
}

// ---------------------------------------------------------------- math
__device__ __forceinline__ float logcosh(float x) {
  float ax = fabsf(x);
  return ax + log1pf(expf(-2.0f * ax)) - 0.69314718055994531f;
}
__device__ __forceinline__ double logcosh(double x) {
  double ax = fabs(x);
  return ax + log1p(exp(-2.0 * ax)) - 0.69314718055994530942;
}

// ---------------------------------------------------------------- XCD-aware block order
// Workgroups are dealt to the 8 XCDs round-robin (block b runs on XCD b % 8).
// Remapping b to x * per + min(x, rem) + b / 8 (x = b % 8) gives each XCD a
// contiguous range of virtual blocks, so data that neighbouring virtual
// blocks share (cache lines of per-chain streams, row panels) stays in one
// XCD's L2.  A bijection of [0, nblocks).
__device__ __forceinline__ int64_t xcd_block(int64_t b, int64_t nblocks) {
  const int64_t per = nblocks / 8, rem = nblocks % 8, x = b % 8, loc = b / 8;
  return x * per + (x < rem ? x : rem) + loc;
}

// ---------------------------------------------------------------- Philox4x32-10
struct u32x4 {
  uint32_t x, y, z, w;
};

__host__ __device__ __forceinline__ u32x4 philox4x32_10(u32x4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    if (r > 0) {
      k0 += 0x9E3779B9u;
      k1 += 0xBB67AE85u;
    }
    uint64_t p0 = (uint64_t)0xD2511F53u * c.x;
    uint64_t p1 = (uint64_t)0xCD9E8D57u * c.z;
    uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
    uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
    c = u32x4{hi1 ^ c.y ^ k0, lo1, hi0 ^ c.w ^ k1, lo0};
  }
  return c;
}

// multiply-shift map of a 32-bit word to [0, n)
__host__ __device__ __forceinline__ uint32_t bounded(uint32_t w, uint32_t n) {
  return (uint32_t)(((uint64_t)w * (uint64_t)n) >> 32);
}

// u = ((w2 << 32 | w3) >> 11) * 2^-53 in [0, 1)
__host__ __device__ __forceinline__ double words_to_uniform(uint32_t w2, uint32_t w3) {
  uint64_t v = ((uint64_t)w2 << 32) | (uint64_t)w3;
  return (double)(v >> 11) * 1.1102230246251565404e-16;
}

// log(u) of the acceptance test (metropolis.py:291-322) in FP64, kept out of
// line: inlined, the constants of FP64 log1p would be hoisted into VGPRs for
// the whole kernel
static __device__ __noinline__ double accept_threshold(uint32_t w2, uint32_t w3) {
  return log1p(-words_to_uniform(w2, w3));
}

constexpr uint32_t TAG_SWEEP = 0x51A7u;
constexpr uint32_t TAG_INIT = 0x1D17u;

// ---------------------------------------------------------------- proposals
// Picks the connected move of one chain.  Spins of the chain live in `sl`
// (LDS, N bytes).  Called by all 64 lanes of a wave with uniform arguments;
// returns the flipped sites (fa, fb; fb = -1 if one site) with `updated`
// false for no-op moves (swap of equal spins / padded neighbour / no hopping
// site).  n_hop is the number of sites holding `hopping` (conserved).
__device__ __forceinline__ void propose_move(int kind, const int8_t* sl, int N, const int32_t* nbr,
                                             int width, int hopping, int n_hop, uint32_t w0, uint32_t w1,
                                             int lane, int& fa, int& fb, bool& updated) {
  if (kind == QTX_LOCALFLIP) {
    fa = (int)bounded(w0, (uint32_t)N);
    fb = -1;
    updated = true;
    return;
  }
  fa = -1;
  fb = -1;
  updated = false;
  if (n_hop <= 0) return;
  uint32_t k = bounded(w0, (uint32_t)n_hop);
  int site = -1;
  for (int base = 0; base < N; base += WAVE) {
    int i = base + lane;
    bool is_hop = (i < N) && (sl[i] == hopping);
    uint64_t m = __ballot(is_hop);
    uint32_t cnt = (uint32_t)__popcll(m);
    if (k < cnt) {
      uint64_t below = (lane == 0) ? 0ull : (m & ((~0ull) >> (64 - lane)));
      bool hit = is_hop && ((uint32_t)__popcll(below) == k);
      uint64_t hm = __ballot(hit);
      site = base + (__ffsll((unsigned long long)hm) - 1);
      break;
    }
    k -= cnt;
  }
  if (site < 0) return;
  uint32_t slot = bounded(w1, (uint32_t)width);
  int nb = nbr[site * width + (int)slot];
  if (nb < 0) nb = site;
  int8_t a = sl[site], b = sl[nb];
  if (nb == site || a == b) return;
  fa = site;
  fb = nb;
  updated = true;
}

// the sites of sl that hold `hopping`, in order, into pos (wave-cooperative LDS);
// returns their number
__device__ __forceinline__ int list_sites(const int8_t* sl, int N, int hopping, uint16_t* pos, int lane) {
  int n = 0;
  for (int base = 0; base < N; base += WAVE) {
    const int i = base + lane;
    const bool is_hop = (i < N) && (sl[i] == hopping);
    const uint64_t m = __ballot(is_hop);
    if (is_hop) pos[n + __popcll(m & ((1ull << lane) - 1))] = (uint16_t)i;
    n += __popcll(m);
  }
  wave_lds_fence();
  return n;
}

// ---------------------------------------------------------------- operator tables
__device__ __forceinline__ double diag_energy(const qtx_ham& H, const int8_t* sl, int lane) {
  double acc = 0.0;
  for (int t = lane; t < H.ndiag; t += WAVE) {
    int kind = H.diag_kind[t];
    double c = H.diag_c[t];
    if (kind == 0)
      acc += c * (double)(sl[H.diag_a[t]] * sl[H.diag_b[t]]);
    else if (kind == 1)
      acc += c * (double)sl[H.diag_a[t]];
    else
      acc += c;
  }
  return wave_sum(acc);
}

__device__ __forceinline__ bool cand_valid(const qtx_ham& H, const int8_t* sl, int k) {
  int a = H.off_a[k], b = H.off_b[k];
  int ra = H.off_ra[k], rb = H.off_rb[k];
  bool ok = (ra == 0) || (sl[a] == ra);
  if (b >= 0) ok = ok && ((rb == 0) || (sl[b] == rb));
  return ok;
}

}  // namespace qtx
