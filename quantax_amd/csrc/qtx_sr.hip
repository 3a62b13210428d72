// SR / MinSR: Omean, Ebar, the MFMA Gram of Obar, rocSOLVER Cholesky / eigh,
// the update vector and the guarded parameter update.
//
// Obar = (O - mean) * sqrt(r / ns) is never materialised: the Gram kernel
// centres each O tile in FP64 while staging it into LDS (then rounds to FP32
// or splits it into bf16 hi/lo), and the update vector x = Obar^T y reads O
// once more with FP64 accumulation.
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <cmath>
#include <cstdlib>
#include <string>
#include <vector>

#include "common.hpp"

namespace qtx {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v4d __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------- helpers
__global__ void fill_f64_kernel(double* p, int64_t n, double v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void fill_i32_kernel(int32_t* p, int64_t n, int32_t v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Column sums over a chunk of rows, accumulated with FP64 atomics:
//   W = false: out_k += sum_s O_sk
//   W = true:  out_k += sum_s (O_sk - mean_k) sqrt(r_s inv_ns) y_s
// HBM-bound: every element is read once.  A lane takes four neighbouring
// columns (one load that needs only the element's own alignment), 2^lg lanes a
// row (64, fewer where np <= 128, so that narrow rows fill the wave too), CS_ROWS
// rows per lane in flight, the last ones of a chunk masked; the rows'
// weights are made once, in LDS, CS_PART at a time.  The sums leave by one column
// per thread: an atomic of a wave touches 512 bytes, where a lane's four columns
// one after another touched 2 KB each time.
// us, means of f32 (one column per thread and row before | this): 4096 x 40400 204 |
// 118, 4096 x 5000 41 | 19, 16384 x 1000 40 | 17, 65536 x 256 132 | 17, 100000 x 8 58 |
// 14, 16 x 1000000 24 | 20, 1024 x 272 17.5 | 13.5.
constexpr int CS_COLS = 256, CS_ROWS = 8, CS_MIN = 16, CS_CHUNKS = 128, CS_PART = 2048;
template <typename TI, bool W>
__global__ __launch_bounds__(256) void colsum_kernel(const TI* __restrict__ O, const double* __restrict__ mean,
                                                     const double* __restrict__ r, const double* __restrict__ y,
                                                     int64_t ns, int64_t np, int64_t rows_per_chunk, int lg,
                                                     double inv_ns, double* __restrict__ out) {
  typedef TI vt4 __attribute__((ext_vector_type(4), aligned(sizeof(TI))));
  __shared__ double ws[W ? CS_PART : 1];
  __shared__ double red[4][CS_COLS];
  const int tid = threadIdx.x, lane = tid % WAVE, q = tid / WAVE;
  const int cl = lane & ((1 << lg) - 1), rw = WAVE >> lg;  // column group of the lane, rows of a wave
  const int first = q * rw + (lane >> lg), step = 4 * rw;
  const int64_t k0 = (int64_t)blockIdx.x * CS_COLS, k = k0 + 4 * cl;
  const int64_t rc = (int64_t)blockIdx.y * rows_per_chunk;
  const int64_t re = rc + rows_per_chunk < ns ? rc + rows_per_chunk : ns;
  const int cols = (int)(k + 4 <= np ? 4 : k < np ? np - k : 0);
  double acc[4] = {0, 0, 0, 0}, m[4] = {0, 0, 0, 0};
  if (W)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (c < cols) m[c] = mean[k + c];
  for (int64_t r0 = rc; r0 < re; r0 += CS_PART) {
    const int rows = (int)(re - r0 < CS_PART ? re - r0 : CS_PART);
    if (W) {
      if (r0 > rc) __syncthreads();  // the last part's weights have been used
      for (int s = tid; s < rows; s += 256) ws[s] = y[r0 + s] * sqrt((r ? r[r0 + s] : 1.0) * inv_ns);
      __syncthreads();
    }
    const TI* p = O + r0 * np + k;
    if (cols == 4) {
      int s = first;
      for (; s + step * (CS_ROWS - 1) < rows; s += step * CS_ROWS) {
        vt4 v[CS_ROWS];
#pragma unroll
        for (int i = 0; i < CS_ROWS; ++i) v[i] = *reinterpret_cast<const vt4*>(p + (s + step * i) * np);
#pragma unroll
        for (int i = 0; i < CS_ROWS; ++i)
#pragma unroll
          for (int c = 0; c < 4; ++c) acc[c] += W ? ((double)v[i][c] - m[c]) * ws[s + step * i] : (double)v[i][c];
      }
      if (s < rows) {
        vt4 v[CS_ROWS];
#pragma unroll
        for (int i = 0; i < CS_ROWS; ++i)
          v[i] = *reinterpret_cast<const vt4*>(p + (s + step * i < rows ? s + step * i : s) * np);
#pragma unroll
        for (int i = 0; i < CS_ROWS; ++i)
          if (s + step * i < rows)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[c] += W ? ((double)v[i][c] - m[c]) * ws[s + step * i] : (double)v[i][c];
      }
    } else if (cols > 0) {
#pragma unroll 4
      for (int s = first; s < rows; s += step)
#pragma unroll
        for (int c = 0; c < 3; ++c)
          if (c < cols) acc[c] += W ? ((double)p[s * np + c] - m[c]) * ws[s] : (double)p[s * np + c];
    }
  }
  for (int d = 1 << lg; d < WAVE; d *= 2)  // over the rows of a wave
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] += __shfl_xor(acc[c], d, WAVE);
  if (lane < 1 << lg)
#pragma unroll
    for (int c = 0; c < 4; ++c) red[q][4 * cl + c] = acc[c];
  __syncthreads();
  // one column per thread: neighbouring atomics
  if (tid < 4 << lg && k0 + tid < np) atomicAdd(out + k0 + tid, red[0][tid] + red[1][tid] + red[2][tid] + red[3][tid]);
}

// rows per chunk, the grid and lg: workgroups of at least CS_MIN wave rows, eight per
// CU, but at most CS_CHUNKS of them, whose atomics on one sum wait for each other (us
// with 32 | 64 | 128 | 256: 1000000 x 3 41 | 24 | 15 | 14, 65536 x 256 39 | 23 | 17 | 19,
// 16384 x 1000 17 | 16 | 17 | 17)
static int64_t colsum_rows(int64_t ns, int64_t np, dim3& g, int& lg) {
  lg = 0;
  while (lg < 6 && (4 << lg) < np) ++lg;
  const int64_t gx = (np + CS_COLS - 1) / CS_COLS, least = (int64_t)CS_MIN * (WAVE >> lg);
  const int64_t fill = std::min<int64_t>(CS_CHUNKS, std::max<int64_t>(1, 2048 / gx));
  const int64_t chunks = std::min<int64_t>(fill, (ns + least - 1) / least);
  const int64_t rpc = (ns + chunks - 1) / chunks;
  g = dim3((unsigned)gx, (unsigned)((ns + rpc - 1) / rpc));
  return rpc;
}

__global__ void scale_f64_kernel(double* p, int64_t n, double a) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] *= a;
}

// single-block: energy, VarE and Ebar (sr.py:180-195)
__global__ __launch_bounds__(1024) void ebar_kernel(const double* __restrict__ E, const double* __restrict__ r,
                                                    int64_t ns, double* __restrict__ ebar, double* __restrict__ out2) {
  __shared__ double red[3][16];
  int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE, nw = blockDim.x / WAVE;
  double s_er = 0, s_e = 0;
  for (int64_t i = tid; i < ns; i += blockDim.x) {
    double ri = r ? r[i] : 1.0;
    s_er += E[i] * ri;
    s_e += E[i];
  }
  s_er = wave_sum(s_er);
  s_e = wave_sum(s_e);
  if (lane == 0) {
    red[0][wv] = s_er;
    red[1][wv] = s_e;
  }
  __syncthreads();
  double tot_er = 0, tot_e = 0;
  for (int w = 0; w < nw; ++w) {
    tot_er += red[0][w];
    tot_e += red[1][w];
  }
  double Emean = tot_er / (double)ns, Eplain = tot_e / (double)ns;
  double s_v = 0;
  for (int64_t i = tid; i < ns; i += blockDim.x) {
    double ri = r ? r[i] : 1.0;
    double d = E[i] - Emean;
    s_v += d * d * ri;
    ebar[i] = (E[i] - Eplain) * sqrt(ri / (double)ns);
  }
  s_v = wave_sum(s_v);
  __syncthreads();
  if (lane == 0) red[2][wv] = s_v;
  __syncthreads();
  if (tid == 0) {
    double tv = 0;
    for (int w = 0; w < nw; ++w) tv += red[2][w];
    out2[0] = Emean;
    out2[1] = tv / (double)ns;
  }
}

// single block: out[0] = 1 if every r_i is one, else 0
__global__ __launch_bounds__(1024) void all_ones_kernel(const double* __restrict__ r, int64_t n,
                                                        double* __restrict__ out) {
  bool other = false;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) other |= !(r[i] == 1.0);
  const int any = __syncthreads_or(other ? 1 : 0);
  if (threadIdx.x == 0) out[0] = any ? 0.0 : 1.0;
}

// ---------------------------------------------------------------- Gram T = A A^T
// A = Obar (n x np) from O rows; only tiles with bi >= bj are computed and
// mirrored.  Output T is FP64 (n x n, symmetric).
constexpr int GT = 128;  // tile of the split-bf16 Gram

__device__ __forceinline__ void tile_of(int bid, int& bi, int& bj) {
  // bid -> (bi, bj) with bj <= bi, row-major over the lower triangle
  int b = (int)((sqrt(8.0 * (double)bid + 1.0) - 1.0) * 0.5);
  while ((b + 1) * (b + 2) / 2 <= bid) ++b;
  while (b * (b + 1) / 2 > bid) --b;
  bi = b;
  bj = bid - b * (b + 1) / 2;
}

// lower-triangle tile t of the XCD-contiguous order: workgroups are dealt to
// the 8 XCDs round-robin, so block b runs on XCD b % 8; giving each XCD a
// contiguous run of tiles (shared row panels) keeps them in its L2
__device__ __forceinline__ int xcd_tile(int bid, int ntiles) {
  const int per = ntiles / 8, rem = ntiles % 8, x = bid % 8, loc = bid / 8;
  return x * per + (x < rem ? x : rem) + loc;
}

// lower-triangle tile (bi, bj) of an mt x mt tile grid from its index t in the
// order of 8 x 8 super-blocks (row-major over the triangle of super-blocks,
// row-major inside each): tiles that run together share few row panels
__device__ __forceinline__ void super_tile_of(int t, int mt, int& bi, int& bj) {
  const int full = mt / 8;  // complete super-rows; super-row R starts at tile 32 R^2 + 4 R
  int R = (int)((sqrt(16.0 + 128.0 * (double)t) - 4.0) / 64.0);
  while (32LL * (R + 1) * (R + 1) + 4LL * (R + 1) <= t) ++R;
  while (32LL * R * R + 4LL * R > t) --R;
  if (R > full) R = full;
  const int rem = t - (32 * R * R + 4 * R);
  const int h = R < full ? 8 : mt - 8 * full;  // tile rows of this super-row
  if (rem < 8 * h * R) {
    const int sb = rem / (8 * h), in = rem - sb * 8 * h;
    bi = 8 * R + in / 8;
    bj = 8 * sb + in % 8;
  } else {
    int a, b;
    tile_of(rem - 8 * h * R, a, b);
    bi = 8 * R + a;
    bj = 8 * R + b;
  }
}

// FP64 / FP32 Gram on 16x16x4 MFMA.  The FP64 matrix pipe takes 64 cycles per
// instruction, so LDS and L2 have room for a small tile: 64 x 64 per
// workgroup (four waves of 32 x 32), four workgroups per CU; a 128 x 128 tile
// would leave the last round of a 4096-row Gram 69 % full.  A thread stages
// four consecutive columns of one row of each operand per 16-column chunk: one
// four-element load of O (which needs only the element's own alignment, so any
// np takes it), fetched one chunk ahead into registers and centred in FP64,
// then written to the other of two LDS
// buffers: one barrier per chunk.  FP64, 4096 x 40400: 44.3 -> 11.7 ms; 4096 x 34952: 38.3
// -> 10.2 ms; 16384 x 34952: 331 -> 154 ms (60 TFLOP/s, a library f64 GEMM
// reaches 73).  The matrix pipe is busy 80 % of the time (SQ counters); the
// FP64 conversions and subtractions, one per MFMA, are most of the rest.
constexpr int GN_T = 64;    // tile
constexpr int GN_KC = 16;   // columns per chunk
constexpr int GN_LD = GN_KC + 1;

// one S x S tile (64 or 32) at (i0, j0) by four waves of S/2 x S/2; As, Bs:
// 2 S GN_LD elements each
template <typename TI, int G, int S, typename ST>
__device__ __forceinline__ void gram_nt_tile(const TI* __restrict__ O, const double* __restrict__ mean,
                                             const double* __restrict__ r, int64_t n, int64_t np, double inv_ns,
                                             int64_t i0, int64_t j0, ST* As, ST* Bs, double* __restrict__ T) {
  constexpr int NB = S / 32;  // 16 x 16 blocks per wave and side
  using ACC = typename std::conditional<G == QTX_GRAM_FP64, v4d, v4f>::type;
  typedef TI vt4 __attribute__((ext_vector_type(4), aligned(sizeof(TI))));
  const int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE;
  const int wr = (wv / 2) * (S / 2), wc = (wv % 2) * (S / 2);  // wave's sub-tile origin
  // staging: columns 4 (tid % 4) .. + 3 of one row; S = 64: row tid / 4 of both
  // operands, S = 32: row tid / 4 % 32 of the first (tid < 128) or the second.
  // Rows past n repeat row n - 1 (their outputs are not stored)
  const int srow = tid / 4 % S, sk = (tid % 4) * 4;
  const bool second = S == 32 && tid >= 128;
  const int64_t ra = i0 + srow < n ? i0 + srow : n - 1, rb = j0 + srow < n ? j0 + srow : n - 1;
  const TI* pa = O + (second ? rb : ra) * np;
  const TI* pb = O + rb * np;
  ST* sa = (second ? Bs : As) + srow * GN_LD + sk;
  ST* sb = Bs + srow * GN_LD + sk;
  // FP32: the row factors go to the staged values, which keeps the products of
  // large O in range (2 to 4 % of its time); FP64: to the sums
  constexpr bool SHADOW = (G != QTX_GRAM_FP64);
  const double fa = SHADOW ? sqrt((r ? r[second ? rb : ra] : 1.0) * inv_ns) : 1.0;
  const double fb = SHADOW ? sqrt((r ? r[rb] : 1.0) * inv_ns) : 1.0;
  TI av[4], bv[4];
  double mv[4];
  auto fetch = [&](int64_t k0) {
    const int64_t k = k0 + sk;
    if (k + 3 < np) {
      const vt4 x = *reinterpret_cast<const vt4*>(pa + k);
      vt4 y;
      if (S == 64) y = *reinterpret_cast<const vt4*>(pb + k);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        av[q] = x[q];
        if (S == 64) bv[q] = y[q];
        mv[q] = mean[k + q];
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bool ok = k + q < np;
        av[q] = ok ? pa[k + q] : TI(0);
        if (S == 64) bv[q] = ok ? pb[k + q] : TI(0);
        mv[q] = ok ? mean[k + q] : 0.0;
      }
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const double x = (double)av[q] - mv[q];
      sa[buf * S * GN_LD + q] = (ST)(SHADOW ? x * fa : x);
      if (S == 64) {
        const double y = (double)bv[q] - mv[q];
        sb[buf * S * GN_LD + q] = (ST)(SHADOW ? y * fb : y);
      }
    }
  };

  ACC acc[NB][NB];
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[a][b] = ACC{0, 0, 0, 0};
  // the FP32 mode flushes its MFMA accumulators into FP64 every FLUSH chunks
  // (256 columns), so the rounding error does not grow with np
  constexpr int FLUSH = 256 / GN_KC;
  v4d dacc[SHADOW ? NB : 1][SHADOW ? NB : 1];
  if constexpr (SHADOW) {
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b) dacc[a][b] = v4d{0, 0, 0, 0};
  }

  const int nchunks = (int)((np + GN_KC - 1) / GN_KC);
  fetch(0);
  stage(0);
  __syncthreads();
  for (int c = 0; c < nchunks; ++c) {
    const ST* Ac = As + (c & 1) * S * GN_LD;
    const ST* Bc = Bs + (c & 1) * S * GN_LD;
    if (c + 1 < nchunks) fetch((int64_t)(c + 1) * GN_KC);
#pragma unroll
    for (int ks = 0; ks < GN_KC; ks += 4) {
      ST af[NB], bf[NB];
#pragma unroll
      for (int a = 0; a < NB; ++a) {
        af[a] = Ac[(wr + a * 16 + lane % 16) * GN_LD + ks + lane / 16];
        bf[a] = Bc[(wc + a * 16 + lane % 16) * GN_LD + ks + lane / 16];
      }
#pragma unroll
      for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          if constexpr (G == QTX_GRAM_FP64)
            acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[a], bf[b], acc[a][b], 0, 0, 0);
          else
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[a], bf[b], acc[a][b], 0, 0, 0);
        }
    }
    if constexpr (SHADOW) {
      if ((c + 1) % FLUSH == 0 || c + 1 == nchunks) {
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
          for (int b = 0; b < NB; ++b) {
#pragma unroll
            for (int q = 0; q < 4; ++q) dacc[a][b][q] += (double)acc[a][b][q];
            acc[a][b] = ACC{0, 0, 0, 0};
          }
      }
    }
    // the other buffer was last read before the previous barrier
    if (c + 1 < nchunks) stage((c + 1) & 1);
    __syncthreads();
  }
  // store, column lane%16 of each 16x16 block; rows of element q:
  //   f32 MFMA: 4 * (lane / 16) + q ;  f64 MFMA: lane / 16 + 4 * q
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int rq = (G == QTX_GRAM_FP64) ? (lane / 16 + 4 * q) : (4 * (lane / 16) + q);
        const int64_t gi = i0 + wr + a * 16 + rq;
        const int64_t gj = j0 + wc + b * 16 + lane % 16;
        // off-diagonal tiles are mirrored; inside diagonal tiles the lower
        // triangle is written to both halves so T is exactly symmetric
        if (gi < n && gj < n && (i0 != j0 || gi >= gj)) {
          double v;
          if constexpr (SHADOW)
            v = dacc[a][b][q];
          else
            v = acc[a][b][q] * (r ? sqrt(r[gi]) * sqrt(r[gj]) * inv_ns : inv_ns);
          T[gi * n + gj] = v;
          T[gj * n + gi] = v;
        }
      }
}

// 32 CUs per XCD take a tile each at a time (four resident at once, so the last
// ones of an XCD's run would end alone on their CUs, one wave per SIMD).  Where
// at most 16 tiles are left over after whole rounds, those are dealt out as 32 x
// 32 quarters, with the same sums: 4096 x 40400 (260 tiles per XCD) 12.9 -> 11.7
// ms, 4096 x 34952 11.2 -> 10.2 ms.
// Few rows (less than a round per XCD) spread over four times the CUs.
__host__ __device__ inline int gram_whole(int per) { return per % 32 <= 16 ? per / 32 * 32 : per; }

template <typename TI, int G>
__global__ __launch_bounds__(256, 4) void gram_nt_kernel(const TI* __restrict__ O, const double* __restrict__ mean,
                                                         const double* __restrict__ r, int64_t n, int64_t np,
                                                         double inv_ns, int ntiles, double* __restrict__ T) {
  using ST = typename std::conditional<G == QTX_GRAM_FP64, double, float>::type;
  __shared__ ST As[2 * GN_T * GN_LD];
  __shared__ ST Bs[2 * GN_T * GN_LD];
  const int x = blockIdx.x % 8, loc = blockIdx.x / 8, per = (ntiles + 7) / 8, whole = gram_whole(per);
  const int tile = loc < whole ? loc : whole + (loc - whole) / 4;
  const int first = xcd_tile(x, ntiles), mine = ntiles / 8 + (x < ntiles % 8 ? 1 : 0);
  if (tile >= mine) return;
  int bi, bj;
  super_tile_of(first + tile, (int)((n + GN_T - 1) / GN_T), bi, bj);
  int64_t i0 = (int64_t)bi * GN_T, j0 = (int64_t)bj * GN_T;
  if (loc < whole) {
    gram_nt_tile<TI, G, 64>(O, mean, r, n, np, inv_ns, i0, j0, As, Bs, T);
  } else {
    i0 += (loc - whole) / 2 % 2 * 32;
    j0 += (loc - whole) % 2 * 32;
    if (i0 < j0 || i0 >= n || j0 >= n) return;  // above the diagonal, or past the end
    gram_nt_tile<TI, G, 32>(O, mean, r, n, np, inv_ns, i0, j0, As, Bs, T);
  }
}

// ---------------------------------------------------------------- split-bf16 Gram
// Pre-pass: Obar = (O - mean) sqrt(r / ns) in FP64, rounded to FP32 x and
// split into bf16 parts hi = bf16(x), lo = bf16(x - hi): per row, 32 hi then their
// 32 lo (one 128-byte line per K step), rows padded to a multiple of GT and K to
// a multiple of G3_KPAD (zeros).  The Gram kernel then streams the parts straight
// into LDS and does only MFMA work: T_ij = sum_k lo_i hi_j + hi_i lo_j + hi_i hi_j
// (lo * lo dropped).
constexpr int G3_KC = 32;            // K per LDS stage (one 16x16x32 MFMA step)
constexpr int G3_FLUSH = 8;          // stages per FP32 -> FP64 flush (256 K)
constexpr int G3_ROW = 2 * G3_KC * 2;     // bytes of a row's hi and lo parts of one stage (a 128-byte line)
constexpr int G3_OPER = GT * G3_ROW;      // bytes of one operand of one stage (16 KB)
constexpr int G3_KPAD = 64;
// From this many tile rows on the super-blocks are dealt to the XCDs one by one:
// the eight that run together then share their row panels, and the last-level
// cache serves what the L2s miss (16384 x 34952: 38.9 -> 37.2 ms, 32768 x 286976:
// 1472 -> 1429).  Below, an XCD takes a contiguous run of tiles: few super-blocks
// do not divide evenly (64 tile rows: 12 % more tiles on one XCD than on average).
constexpr int G3_DEAL = 96;

static inline int64_t g3_rows(int64_t n) { return (n + GT - 1) / GT * GT; }
static inline int64_t g3_kpad(int64_t np) { return (np + G3_KPAD - 1) / G3_KPAD * G3_KPAD; }
static inline size_t g3_bytes(int64_t n, int64_t np) { return (size_t)g3_rows(n) * g3_kpad(np) * 2 * sizeof(__bf16); }

// Eight columns per thread: one row factor for them, two loads that need only the
// element's own alignment, one 16-byte store per part.  HBM-bound: 16384 x 34952
// 1.57 -> 1.13 ms (one column, a square root and two 2-byte stores per thread
// before).  Grid-stride over (row, 2048-column block) pairs: a launch's work-item
// count is a 32-bit quantity, and rows * kpad passes 2^32 at 32768 x 286976.
constexpr int SP_COLS = 8;
template <typename TI>
__global__ __launch_bounds__(256) void split_bf16x3_kernel(const TI* __restrict__ O, const double* __restrict__ mean,
                                                           const double* __restrict__ r, int64_t n, int64_t np,
                                                           int64_t kpad, int64_t bpr, int64_t nblocks, double inv_ns,
                                                           __bf16* __restrict__ HL) {
  typedef TI vt4 __attribute__((ext_vector_type(4), aligned(sizeof(TI))));
  for (int64_t blk = blockIdx.x; blk < nblocks; blk += gridDim.x) {
    const int64_t row = blk / bpr;
    const int64_t k = ((blk % bpr) * 256 + threadIdx.x) * SP_COLS;
    if (k >= kpad) continue;
    TI o[SP_COLS];
    double m[SP_COLS];
    const TI* p = O + row * np + k;
    const bool in = row < n;
    if (in && k + SP_COLS <= np) {
      const vt4 x = *reinterpret_cast<const vt4*>(p), y = *reinterpret_cast<const vt4*>(p + 4);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        o[c] = x[c];
        o[c + 4] = y[c];
      }
#pragma unroll
      for (int c = 0; c < SP_COLS; ++c) m[c] = mean[k + c];
    } else {
#pragma unroll
      for (int c = 0; c < SP_COLS; ++c) {
        const bool ok = in && k + c < np;
        o[c] = ok ? p[c] : TI(0);
        m[c] = ok ? mean[k + c] : 0.0;
      }
    }
    const double f = sqrt((r && in ? r[row] : 1.0) * inv_ns);
    v8bf hi, lo;
#pragma unroll
    for (int c = 0; c < SP_COLS; ++c) {
      float x = (float)(((double)o[c] - m[c]) * f);
      asm("" : "+v"(x));  // rounded to single precision first: not folded into FP64 -> bf16
      hi[c] = (__bf16)x;
      lo[c] = (__bf16)(x - (float)hi[c]);
    }
    __bf16* q = HL + 2 * (row * kpad + k / G3_KC * G3_KC) + k % G3_KC;
    *reinterpret_cast<v8bf*>(q) = hi;
    *reinterpret_cast<v8bf*>(q + G3_KC) = lo;
  }
}

typedef __attribute__((address_space(3))) void lds_void;

// 128 x 128 tile, 4 waves (2 x 2, 64 x 64 each), two workgroups per CU so that one
// multiplies while the other waits.  Operands move HBM -> LDS by LDS DMA
// (global_load_lds_dwordx4: lane l of a wave writes 16 bytes at the wave's LDS
// base + 16 l), two 32 KB stages so chunk c + 1 is in flight while chunk c is
// multiplied.  A row of a stage is one line, hi and lo of 32 K; its 16-byte
// segment s (hi 0-3, lo 4-7) sits in slot s ^ (r & 7), so the MFMA fragment reads
// (16 rows, one segment) hit 8 distinct slots per 8 lanes: no bank conflicts.
// The stage barriers are raw s_barrier with explicit vmcnt waits: a
// __syncthreads() fence would drain the next chunk's DMA as well.
// Bound by L2 misses at large n: the 64 tiles an XCD runs together (an 8 x 8
// super-block) drift apart in K by more than its L2 holds, 154 GB at 4.3 TB/s for
// 16384 x 34952, where 37 GB would do.  16384 x 34952 with the pass above: 41.7 ->
// 36.5 ms; 8192: 9.8 ms, 4096: 3.9 -> 2.9 ms (one workgroup per CU with separate
// planes and K = 64 stages before; half-line stages, 64 bytes per row and plane,
// took 46.5 ms at 16384).
__global__ __launch_bounds__(256, 2) void gram_bf16x3_kernel(const __bf16* __restrict__ HL, int64_t n, int64_t kpad,
                                                             int ntiles, double* __restrict__ T) {
  __shared__ __attribute__((aligned(16))) char smem[2 * 2 * G3_OPER];
  int bi, bj;
  const int mt = (int)((n + GT - 1) / GT);
  if (mt < G3_DEAL) {
    super_tile_of(xcd_tile(blockIdx.x, ntiles), mt, bi, bj);
  } else {
    const int x = blockIdx.x % 8, loc = blockIdx.x / 8, in = loc % 64;
    int R, C;
    tile_of(loc / 64 * 8 + x, R, C);
    bi = in / 8;
    bj = in % 8;
    if (R == C) {
      if (in >= 36) return;
      tile_of(in, bi, bj);
    }
    bi += 8 * R;
    bj += 8 * C;
    if (bi >= mt) return;
  }
  const int64_t i0 = (int64_t)bi * GT, j0 = (int64_t)bj * GT;
  const int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE;
  const int wr = (wv / 2) * 64, wc = (wv % 2) * 64;
  // wave w fetches rows 64 (w % 2) .. of the first (w < 2) or the second operand.
  // One DMA instruction covers rows 8 q .. 8 q + 7: lane l -> row 8 q + l / 8, slot
  // l % 8, which holds logical segment (l % 8) ^ (l / 8)
  const int lrow = lane / 8, lseg = (lane % 8) ^ (lane / 8);
  const __bf16* src = HL + 2 * ((wv < 2 ? i0 : j0) + 64 * (wv % 2) + lrow) * kpad + lseg * 8;
  auto issue = [&](int64_t k0, int stage) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const __bf16* g = src + 2 * (q * 8 * kpad + k0);
      char* dst = smem + (stage * 2 + wv / 2) * G3_OPER + (wv % 2) * (G3_OPER / 2) + q * 1024;
      __builtin_amdgcn_global_load_lds((const void*)g, (lds_void*)dst, 16, 0, 0);
    }
  };

  v4f acc[4][4];
  v4d dacc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      acc[a][b] = v4f{0, 0, 0, 0};
      dacc[a][b] = v4d{0, 0, 0, 0};
    }
  const int nchunks = (int)(kpad / G3_KC);
  issue(0, 0);
  if (nchunks > 1) issue(G3_KC, 1);
  for (int c = 0; c < nchunks; ++c) {
    // this wave's DMA for chunk c is done (8 newer ones may be in flight), then
    // every wave's is
    if (c + 1 < nchunks)
      asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    const char* stg = smem + (c & 1) * 2 * G3_OPER;
    const int hs = ((lane / 16) ^ (lane & 7)) * 16, ls = hs ^ 64;  // slots of hi and lo, the same for every 16-row block
    v8bf bh[4], bl[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const char* row = stg + G3_OPER + (wc + b * 16 + lane % 16) * G3_ROW;
      bh[b] = *(const v8bf*)(row + hs);
      bl[b] = *(const v8bf*)(row + ls);
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const char* row = stg + (wr + a * 16 + lane % 16) * G3_ROW;
      const v8bf ah = *(const v8bf*)(row + hs), al = *(const v8bf*)(row + ls);
      // the three products of a block are 4 MFMAs apart (no back-to-back dependency)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh[b], acc[a][b], 0, 0, 0);
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl[b], acc[a][b], 0, 0, 0);
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh[b], acc[a][b], 0, 0, 0);
    }
    if ((c + 1) % G3_FLUSH == 0 || c + 1 == nchunks) {
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
#pragma unroll
          for (int q = 0; q < 4; ++q) dacc[a][b][q] += (double)acc[a][b][q];
          acc[a][b] = v4f{0, 0, 0, 0};
        }
    }
    // every wave has read this stage (its fragments fed the MFMAs above)
    // before the DMA of chunk c + 2 overwrites it
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (c + 2 < nchunks) issue((int64_t)(c + 2) * G3_KC, c & 1);
  }
  // element q of a 16x16 block: row 4 * (lane / 16) + q, column lane % 16
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t gi = i0 + wr + a * 16 + 4 * (lane / 16) + q;
        const int64_t gj = j0 + wc + b * 16 + lane % 16;
        if (gi < n && gj < n && (bi != bj || gi >= gj)) {
          T[gi * n + gj] = dacc[a][b][q];
          T[gj * n + gi] = dacc[a][b][q];
        }
      }
}

// No use of an accumulator before its MFMA is done, whatever branch follows:
// the distance is kept here, not counted along one path
template <int N>
__device__ __forceinline__ void mfma_settle_f64(v4d* acc) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(acc[i]));
  asm volatile("s_nop 15\n\ts_nop 7" : "+v"(acc[0]));
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(acc[i]));
}

// S = Obar^T Obar (np x np), FP64 (SR branch, ns >= np).  One 16 x 16 tile of
// the lower triangle per workgroup, its 16 waves a part of the samples each (every
// 16th group of four): an MFMA's operands are 16 neighbouring columns
// of four samples, read from O as they lie (no staging, no Obar in memory), TN_U
// steps in flight.  Bound by the FP64 matrix pipe and the L1 (64 B per cycle) once
// there are enough tiles; by the loads' latency with few samples.
// 1024 x 272 f64: 10.7 us (43 with Obar formed and a library DGEMM, which is what
// larger np take in a solve, kGramTnMax).
constexpr int TN_U = 4, TN_W = 16;
template <typename TI>
__global__ __launch_bounds__(WAVE * TN_W) void gram_tn_kernel(const TI* __restrict__ O, const double* __restrict__ mean,
                                                      const double* __restrict__ r, int64_t ns, int64_t np,
                                                      double inv_ns, double* __restrict__ S) {
  __shared__ double red[TN_W - 1][4][WAVE];
  int bi, bj;
  tile_of(blockIdx.x, bi, bj);
  const int lane = threadIdx.x % WAVE, g = lane / 16, m = lane % 16;
  const int q = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int64_t k = 16 * (int64_t)bi + m, l = 16 * (int64_t)bj + m;
  const int64_t kc = k < np ? k : np - 1, lc = l < np ? l : np - 1;  // columns past np: not stored
  const double mk = mean[kc], ml = mean[lc];
  v4d acc[1] = {v4d{0, 0, 0, 0}};
  TI a[2][TN_U], b[2][TN_U];
  double w[2][TN_U];
  auto load = [&](int64_t s0, int p) {  // samples past ns: weight 0
#pragma unroll
    for (int u = 0; u < TN_U; ++u) {
      const int64_t s = s0 + 4 * TN_W * u + 4 * q + g, sc = s < ns ? s : ns - 1;
      a[p][u] = O[sc * np + kc];
      b[p][u] = O[sc * np + lc];
      const double rs = r ? r[sc] : 1.0;
      w[p][u] = s < ns ? (rs < 0.0 ? NAN : rs) * inv_ns : 0.0;  // of a negative factor there is no root
    }
  };
  auto use = [&](int p) {
#pragma unroll
    for (int u = 0; u < TN_U; ++u)
      acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(((double)a[p][u] - mk) * w[p][u], (double)b[p][u] - ml, acc[0], 0,
                                                    0, 0);
  };
  constexpr int STEP = 4 * TN_W * TN_U;
  load(0, 0);
  for (int64_t s0 = 0; s0 < ns; s0 += 2 * STEP) {  // the next part is on its way during this one's products
    load(s0 + STEP, 1);
    use(0);
    load(s0 + 2 * STEP, 0);
    use(1);
  }
  mfma_settle_f64<1>(acc);
  if (q > 0)
#pragma unroll
    for (int v = 0; v < 4; ++v) red[q - 1][v][lane] = acc[0][v];
  __syncthreads();
  if (q > 0) return;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    double x = acc[0][v];
#pragma unroll
    for (int p = 0; p < TN_W - 1; ++p) x += red[p][v][lane];
    const int64_t row = 16 * (int64_t)bi + 4 * v + g;
    if (row < np && l < np && row >= l) {
      S[row * np + l] = x;
      S[l * np + row] = x;
    }
  }
}

// np up to which a solve forms S by gram_tn_kernel (us, it | Obar and DGEMM): 1024 x
// 272 10.7 | 43, 4096 x 272 35 | 137, 8192 x 272 63 | 232, 4096 x 512 94 | 135, 4096
// x 1000 250 | 144, 8192 x 1000 482 | 911, 4096 x 2000 942 | 495.  Many samples do not
// move it, though a tile is one workgroup over all of them (whole shifted solves, ms):
// 65536 x 72 0.45 | 7.3, 262144 x 272 1.7 | 14.9, 65536 x 512 1.4 | 8.0, 1000000 x 8 5.2 | 54
constexpr int64_t kGramTnMax = 512;
// whether the SR branch forms Obar in memory: S of more parameters, the SNR products
static inline bool needs_obar(int64_t np, int mode) { return np > kGramTnMax || (mode & QTX_SOLVE_SNR); }

template <typename TI>
static int launch_gram_tn(hipStream_t st, const TI* O, const double* mean, const double* r, int64_t ns, int64_t np,
                          double* S) {
  const int64_t nt = (np + 15) / 16, tiles = nt * (nt + 1) / 2;
  QTX_REQUIRE(tiles < 0x7fffffff, "Gram too large");
  hipLaunchKernelGGL(gram_tn_kernel<TI>, dim3((unsigned)tiles), dim3(WAVE * TN_W), 0, st, O, mean, r, ns, np,
                     1.0 / (double)ns, S);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

// out[s, k] = (O[s, k] - mean[k]) sqrt(r_s / ns) in FP64 (grid-stride)
template <typename TI>
__global__ void form_obar_kernel(const TI* __restrict__ O, const double* __restrict__ mean,
                                 const double* __restrict__ r, int64_t ns, int64_t np, double inv_ns,
                                 double* __restrict__ out) {
  const int64_t total = ns * np;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t s = e / np, k = e - s * np;
    out[e] = ((double)O[e] - mean[k]) * sqrt((r ? r[s] : 1.0) * inv_ns);
  }
}

// y_s = beta y_s + alpha sqrt(r_s / ns) sum_k (O_sk - mean_k) v_k: the product
// Obar v, one wave per sample row (FP64 accumulation)
template <typename TI>
__global__ __launch_bounds__(256) void obar_matvec_kernel(const TI* __restrict__ O, const double* __restrict__ mean,
                                                          const double* __restrict__ r, int64_t ns, int64_t np,
                                                          double inv_ns, double alpha, const double* __restrict__ v,
                                                          double beta, double* __restrict__ y) {
  const int lane = threadIdx.x % WAVE;
  const int64_t s = (int64_t)blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE;
  if (s >= ns) return;
  const TI* row = O + s * np;
  double a0 = 0.0, a1 = 0.0;
  int64_t k = lane;
  for (; k + WAVE < np; k += 2 * WAVE) {
    a0 += ((double)row[k] - mean[k]) * v[k];
    a1 += ((double)row[k + WAVE] - mean[k + WAVE]) * v[k + WAVE];
  }
  if (k < np) a0 += ((double)row[k] - mean[k]) * v[k];
  const double acc = wave_sum(a0 + a1);
  if (lane == 0) y[s] = (beta == 0.0 ? 0.0 : beta * y[s]) + alpha * sqrt((r ? r[s] : 1.0) * inv_ns) * acc;
}

// O[:, k] *= d_k (grid-stride over the ns * np elements), mean_k *= d_k
template <typename TI>
__global__ void scale_columns_kernel(TI* __restrict__ O, int64_t ns, int64_t np, const double* __restrict__ d) {
  const int64_t total = ns * np;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x)
    O[e] = (TI)((double)O[e] * d[e % np]);
}

__global__ void mul_f64_kernel(double* __restrict__ x, const double* __restrict__ d, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] *= d[i];
}

// single-block: scalars[0] = trace, then T_ii += rshift * trace + ashift
__global__ __launch_bounds__(1024) void shift_diag_kernel(double* __restrict__ T, int64_t n, double rshift,
                                                          double ashift, double* __restrict__ scalars) {
  __shared__ double red[16];
  int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE, nw = blockDim.x / WAVE;
  double acc = 0.0;
  for (int64_t i = tid; i < n; i += blockDim.x) acc += T[i * n + i];
  acc = wave_sum(acc);
  if (lane == 0) red[wv] = acc;
  __syncthreads();
  double tr = 0.0;
  for (int w = 0; w < nw; ++w) tr += red[w];
  double shift = rshift * tr + ashift;
  for (int64_t i = tid; i < n; i += blockDim.x) T[i * n + i] += shift;
  if (tid == 0) scalars[0] = tr;
}

// single block: scale[0] = 2^k with 2^k * max_i |T_ii| in [0.5, 1) (exact scaling)
__global__ __launch_bounds__(1024) void pow2_scale_kernel(const double* __restrict__ T, int64_t n,
                                                          double* __restrict__ scale) {
  __shared__ double red[16];
  int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE, nw = blockDim.x / WAVE;
  double m = 0.0;
  for (int64_t i = tid; i < n; i += blockDim.x) m = fmax(m, fabs(T[i * n + i]));
  m = wave_max(m);
  if (lane == 0) red[wv] = m;
  __syncthreads();
  if (tid == 0) {
    double mx = 0.0;
    for (int w = 0; w < nw; ++w) mx = fmax(mx, red[w]);
    int e = 0;
    if (mx > 0.0 && isfinite(mx)) frexp(mx, &e);  // mx = f * 2^e, f in [0.5, 1)
    scale[0] = ldexp(1.0, -e);
  }
}

__global__ void scale_by_kernel(double* __restrict__ T, int64_t n2, const double* __restrict__ scale) {
  const double sc = scale[0];
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n2; i += (int64_t)gridDim.x * blockDim.x)
    T[i] *= sc;
}

// soft inverse of eigenvalues times rho (solver.py:94-101), single block
__global__ __launch_bounds__(1024) void eig_inv_kernel(const double* __restrict__ vals, int64_t n, double rtol,
                                                       double atol, const double* __restrict__ scale,
                                                       double* __restrict__ rho) {
  const double inv_scale = 1.0 / scale[0];  // eigenvalues of the scaled matrix -> eigenvalues of T
  __shared__ double red[16];
  int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE, nw = blockDim.x / WAVE;
  double m = 0.0;
  for (int64_t i = tid; i < n; i += blockDim.x) m = fmax(m, fabs(vals[i] * inv_scale));
  m = wave_max(m);
  if (lane == 0) red[wv] = m;
  __syncthreads();
  double vmax = 0.0;
  for (int w = 0; w < nw; ++w) vmax = fmax(vmax, red[w]);
  double cut = rtol * vmax + atol;
  for (int64_t i = tid; i < n; i += blockDim.x) {
    double v = vals[i] * inv_scale, va = fabs(v);
    double inv = 0.0;
    if (va > 0.0) {
      double q = cut / va;
      double q2 = q * q;
      inv = 1.0 / (v * (1.0 + q2 * q2 * q2));
    }
    rho[i] *= inv;
  }
}

__global__ void copy_f64_kernel(const double* __restrict__ a, double* __restrict__ b, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

template <typename T>
__global__ __launch_bounds__(256) void finite_check_kernel(const double* __restrict__ step, int64_t n,
                                                           int32_t* __restrict__ ok) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool bad = (i < n) && !isfinite(step[i]);
  if (__any(bad) && (threadIdx.x % WAVE) == 0) atomicAnd(ok, 0);
}

template <typename T>
__global__ __launch_bounds__(256) void apply_update_kernel(T* __restrict__ theta, const double* __restrict__ step,
                                                           double lr, int64_t n, const int32_t* __restrict__ ok) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || *ok == 0) return;
  T d = (T)(lr * step[i]);
  theta[i] = theta[i] - d;
}

// ---------------------------------------------------------------- soft inverse by partial fractions
// The soft inverse of solver.py:94-101, g(v) = 1 / (v (1 + (c/|v|)^6)), equals
// v^5 / (v^6 + c^6).  Its six simple poles p_k = c exp(i pi (2k+1)/6) all have
// residue 1/6, so pairing conjugates
//   g(v) = (1/3) sum_{k=0..2} Re 1 / (v - p_k),
// and g(T) b = (1/3) sum_k Re (T - p_k I)^{-1} b needs no eigendecomposition.
// Each complex system is solved by iterative refinement whose inner solve is
// (T - conj(p) I) ((T - a)^2 + b^2)^{-1}, p = a + ib, with the real SPD
// quadratic factored once by Cholesky; the residual uses T itself, so the
// result has the accuracy of the well-conditioned complex system.

// 16 bytes of a matrix streamed once per pass: a non-temporal load, which
// leaves the caches to the vector operand
typedef double v2d_nt __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double2 stream_load2(const double2* p) {
  const v2d_nt v = __builtin_nontemporal_load(reinterpret_cast<const v2d_nt*>(p));
  return make_double2(v.x, v.y);
}

// One wave's partial sums of row[j] * x[j] over j in [lo, hi): 16-byte loads
// (1 KB per wave instruction; the row's non-temporal) where row and x share
// their 16-byte alignment phase, after peeling one element to reach it;
// 8-byte loads otherwise.  At n = 16384 a triangle pass (1.07 GB) takes
// ~180 us, a full-matrix pass ~330 us (6.5 TB/s).
__device__ __forceinline__ double wave_row_dot(const double* __restrict__ row, const double* __restrict__ x,
                                               int64_t lo, int64_t hi, int lane) {
  double acc = 0.0;
  if (((reinterpret_cast<uintptr_t>(row) ^ reinterpret_cast<uintptr_t>(x)) & 15) == 0) {
    if ((reinterpret_cast<uintptr_t>(row + lo) & 15) && lo < hi) {
      if (lane == 0) acc = row[lo] * x[lo];
      ++lo;
    }
    const double2* r2 = reinterpret_cast<const double2*>(row + lo);
    const double2* x2 = reinterpret_cast<const double2*>(x + lo);
    const int64_t m = (hi - lo) / 2;
    int64_t k = lane;
    for (; k + 3 * WAVE < m; k += 4 * WAVE) {
      const double2 a0 = stream_load2(r2 + k), a1 = stream_load2(r2 + k + WAVE),
                    a2 = stream_load2(r2 + k + 2 * WAVE), a3 = stream_load2(r2 + k + 3 * WAVE);
      const double2 b0 = x2[k], b1 = x2[k + WAVE], b2 = x2[k + 2 * WAVE], b3 = x2[k + 3 * WAVE];
      acc += a0.x * b0.x + a0.y * b0.y + a1.x * b1.x + a1.y * b1.y + a2.x * b2.x + a2.y * b2.y + a3.x * b3.x +
             a3.y * b3.y;
    }
    for (; k < m; k += WAVE) {
      const double2 a0 = stream_load2(r2 + k), b0 = x2[k];
      acc += a0.x * b0.x + a0.y * b0.y;
    }
    if (((hi - lo) & 1) && lane == 0) acc += row[hi - 1] * x[hi - 1];
    return acc;
  }
  int64_t j = lo + lane;
  for (; j + 3 * WAVE < hi; j += 4 * WAVE)
    acc += row[j] * x[j] + row[j + WAVE] * x[j + WAVE] + row[j + 2 * WAVE] * x[j + 2 * WAVE] +
           row[j + 3 * WAVE] * x[j + 3 * WAVE];
  for (; j < hi; j += WAVE) acc += row[j] * x[j];
  return acc;
}

// Y = T X for NV vectors (n x NV, column-major) with T symmetric n x n stored
// in full: one wave per row, coalesced reads of the row, X from cache.
// An HBM stream of T at close to copy bandwidth (library GEMV / GEMM with
// one or two columns reach a fraction of it).
template <int NV>
__global__ __launch_bounds__(256) void matvec_rows_kernel(const double* __restrict__ T, int64_t n,
                                                          const double* __restrict__ X, double* __restrict__ Y) {
  const int lane = threadIdx.x % WAVE;
  const int64_t i = (int64_t)blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE;
  if (i >= n) return;
  const double* row = T + i * n;
  if constexpr (NV == 1) {
    const double s = wave_sum(wave_row_dot(row, X, 0, n, lane));
    if (lane == 0) Y[i] = s;
    return;
  }
  double acc[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) acc[v] = 0.0;
  int64_t j = lane;
  for (; j + 3 * WAVE < n; j += 4 * WAVE) {
    const double t0 = row[j], t1 = row[j + WAVE], t2 = row[j + 2 * WAVE], t3 = row[j + 3 * WAVE];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const double* x = X + v * n + j;
      acc[v] += t0 * x[0] + t1 * x[WAVE] + t2 * x[2 * WAVE] + t3 * x[3 * WAVE];
    }
  }
  for (; j < n; j += WAVE) {
    const double tj = row[j];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] += tj * X[v * n + j];
  }
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const double s = wave_sum(acc[v]);
    if (lane == 0) Y[v * n + i] = s;
  }
}

// sum over the block (every thread gets the total; fixed summation order)
__device__ __forceinline__ double block_sum(double x, double* red) {
  int tid = threadIdx.x, lane = tid % WAVE, wv = tid / WAVE, nw = blockDim.x / WAVE;
  x = wave_sum(x);
  __syncthreads();  // red may still be read by a previous call
  if (lane == 0) red[wv] = x;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < nw; ++w) t += red[w];
  return t;
}

// single block: V[0..n) = hashed start vector / norm, V[n..3n) = 0, beta[0] = 0
__global__ __launch_bounds__(1024) void lanczos_init_kernel(int64_t n, double* __restrict__ V,
                                                            double* __restrict__ beta) {
  __shared__ double red[16];
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    uint64_t z = (uint64_t)i * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;  // splitmix64
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    double v = (double)(z >> 11) * 0x1.0p-52 - 1.0;  // [-1, 1)
    V[i] = v;
    V[n + i] = 0.0;
    V[2 * n + i] = 0.0;
    acc += v * v;
  }
  double inv = 1.0 / sqrt(block_sum(acc, red));
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) V[i] *= inv;
  if (threadIdx.x == 0) beta[0] = 0.0;
}

// single block, after w = T v_j: alpha_j = w.v_j, w -= alpha_j v_j + beta_j v_{j-1},
// one re-orthogonalisation against v_j, beta_{j+1} = |w|, v_{j+1} = w / beta_{j+1}.
// n <= 1024 K (K > 0): the vectors are read once and stay in registers, so the
// block waits for memory once instead of three times (27 -> 16 us at n = 16384,
// 10.3 -> 6 us at 4096); K = 0 takes any n.
template <int K>
__global__ __launch_bounds__(1024) void lanczos_step_kernel(int64_t n, int j, double* __restrict__ w,
                                                            const double* __restrict__ v,
                                                            const double* __restrict__ vp, double* __restrict__ vn,
                                                            double* __restrict__ alpha, double* __restrict__ beta) {
  __shared__ double red[16];
  const double bj = beta[j];
  double a = 0.0, a2 = 0.0, nn = 0.0;
  if constexpr (K > 0) {
    double wr[K], vr[K], pr[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int64_t i = threadIdx.x + 1024 * k;
      wr[k] = i < n ? w[i] : 0.0;
      vr[k] = i < n ? v[i] : 0.0;
      pr[k] = i < n ? vp[i] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) a += wr[k] * vr[k];
    a = block_sum(a, red);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      wr[k] = wr[k] - a * vr[k] - bj * pr[k];
      a2 += wr[k] * vr[k];
    }
    a2 = block_sum(a2, red);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      wr[k] -= a2 * vr[k];
      nn += wr[k] * wr[k];
    }
    nn = sqrt(block_sum(nn, red));
    const double inv = nn > 0.0 ? 1.0 / nn : 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int64_t i = threadIdx.x + 1024 * k;
      if (i < n) vn[i] = wr[k] * inv;
    }
  } else {
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) a += w[i] * v[i];
    a = block_sum(a, red);
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
      double t = w[i] - a * v[i] - bj * vp[i];
      w[i] = t;
      a2 += t * v[i];
    }
    a2 = block_sum(a2, red);
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
      double t = w[i] - a2 * v[i];
      w[i] = t;
      nn += t * t;
    }
    nn = sqrt(block_sum(nn, red));
    const double inv = nn > 0.0 ? 1.0 / nn : 0.0;
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) vn[i] = w[i] * inv;
  }
  if (threadIdx.x == 0) {
    alpha[j] = a + a2;
    beta[j + 1] = nn;
  }
}

// A = T2 - 2a T + c^2 I on the lower triangle (column-major, i >= j), 0 above
__global__ __launch_bounds__(256) void form_quad_kernel(const double* T2,
                                                        const double* __restrict__ T, int64_t n, double two_a,
                                                        double c2, double* A) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n * n; e += (int64_t)gridDim.x * blockDim.x) {
    int64_t j = e / n, i = e - j * n;
    A[e] = (i < j) ? 0.0 : T2[e] - two_a * T[e] + (i == j ? c2 : 0.0);
  }
}

// Shifted Cholesky route for small cutoffs (c < 1e-5 lambda_max, the
// reference default rtol = 1e-12): G = T + (mu / n) 1 1^T - sigma I, lower
// triangle (the upper part zero), factored once; x = T^+ b' is refined against
// T + (mu / n) 1 1^T, which deflates the null direction 1 of the centred MinSR
// Gram (mu = 0 for the SR branch), by conjugate gradients preconditioned
// with that factor.
__global__ __launch_bounds__(256) void form_shifted_kernel(const double* __restrict__ T, int64_t n, double mu_n,
                                                           double sigma, double* __restrict__ G) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n * n; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t j = e / n, i = e - j * n;
    G[e] = (i < j) ? 0.0 : T[e] + mu_n - (i == j ? sigma : 0.0);
  }
}

__device__ double block_sum_1024(double v, double* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x % WAVE, wv = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
  __syncthreads();
  if (lane == 0) red[wv] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < nw; ++w) s += red[w];
  return s;
}

// single block: b' = b - mean(b) 1 (deflate) or b; x = 0; r = z = b'
__global__ __launch_bounds__(1024) void shifted_init_kernel(const double* __restrict__ b, int64_t n, int deflate,
                                                            double* __restrict__ bp, double* __restrict__ x,
                                                            double* __restrict__ r, double* __restrict__ z) {
  __shared__ double red[16];
  double s = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) s += b[i];
  const double mean = deflate ? block_sum_1024(s, red) / (double)n : 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    const double v = b[i] - mean;
    bp[i] = v;
    r[i] = v;
    z[i] = v;
    x[i] = 0.0;
  }
}

// Conjugate gradients on T_d x = b' preconditioned by the factor of
// G = T_d - sigma I (the preconditioned operator is I + sigma G^-1: eigenvalues
// 1 + sigma / (v - sigma), clustered at 1 except for the few v near sigma).
// s[0] holds r.z.  Single-block steps around the library's triangular solves.
// step 1: q = T p (given) + (mu / n) sum(p); alpha = rz / p.q; x += alpha p;
// r -= alpha q; z = r (then z <- G^-1 z by two triangular solves)
__global__ __launch_bounds__(1024) void pcg_step1_kernel(double* __restrict__ q, const double* __restrict__ p,
                                                         int64_t n, double mu_n, double* __restrict__ x,
                                                         double* __restrict__ r, double* __restrict__ z,
                                                         const double* __restrict__ s) {
  __shared__ double red[16];
  double sp = 0.0;
  if (mu_n != 0.0)
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) sp += p[i];
  const double add = (mu_n != 0.0) ? mu_n * block_sum_1024(sp, red) : 0.0;
  double pq = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    const double qi = q[i] + add;
    q[i] = qi;
    pq += p[i] * qi;
  }
  pq = block_sum_1024(pq, red);
  const double alpha = (pq > 0.0 && std::isfinite(pq)) ? s[0] / pq : 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    x[i] += alpha * p[i];
    const double ri = r[i] - alpha * q[i];
    r[i] = ri;
    z[i] = ri;
  }
}

// step 2 (first = 1: p = z): rz' = r.z; beta = rz' / rz; p = z + beta p; s[0] = rz'
__global__ __launch_bounds__(1024) void pcg_step2_kernel(const double* __restrict__ r, const double* __restrict__ z,
                                                         int64_t n, int first, double* __restrict__ p,
                                                         double* __restrict__ s) {
  __shared__ double red[16];
  double rz = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) rz += r[i] * z[i];
  rz = block_sum_1024(rz, red);
  const double beta = (!first && s[0] > 0.0 && std::isfinite(rz)) ? rz / s[0] : 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) p[i] = z[i] + beta * p[i];
  __syncthreads();
  if (threadIdx.x == 0) s[0] = rz;
}

// the true residual of the result: norms <- |b' - T_d x|^2, |x|^2 (Tx given)
__global__ __launch_bounds__(1024) void pcg_check_kernel(const double* __restrict__ bp, const double* __restrict__ Tx,
                                                         const double* __restrict__ x, int64_t n, double mu_n,
                                                         double* __restrict__ norms) {
  __shared__ double red[16];
  double sx = 0.0;
  if (mu_n != 0.0)
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) sx += x[i];
  const double add = (mu_n != 0.0) ? mu_n * block_sum_1024(sx, red) : 0.0;
  double rr = 0.0, xx = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    const double ri = bp[i] - Tx[i] - add;
    rr += ri * ri;
    xx += x[i] * x[i];
  }
  rr = block_sum_1024(rr, red);
  xx = block_sum_1024(xx, red);
  if (threadIdx.x == 0) {
    norms[0] = rr;
    norms[1] = xx;
  }
}

// R = [b, 0], Z = 0   (R, Z: n x 2 column-major)
__global__ void refine_init_kernel(const double* __restrict__ rhs, int64_t n, double* __restrict__ R,
                                   double* __restrict__ Z) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  R[i] = rhs[i];
  R[n + i] = 0.0;
  Z[i] = 0.0;
  Z[n + i] = 0.0;
}

// Z += (T - conj(p)) W with W = A^{-1} R, TW = T W
__global__ void refine_update_kernel(const double* __restrict__ W, const double* __restrict__ TW, int64_t n,
                                     double a, double b, double* __restrict__ Z) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double wr = W[i], wi = W[n + i];
  Z[i] += TW[i] - a * wr - b * wi;
  Z[n + i] += TW[n + i] - a * wi + b * wr;
}

// R = b - (T - p) Z with TZ = T Z
__global__ void refine_residual_kernel(const double* __restrict__ rhs, const double* __restrict__ Z,
                                       const double* __restrict__ TZ, int64_t n, double a, double b,
                                       double* __restrict__ R) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double zr = Z[i], zi = Z[n + i];
  R[i] = rhs[i] - (TZ[i] - a * zr + b * zi);
  R[n + i] = -(TZ[n + i] - a * zi - b * zr);
}

// x (+)= Re Z / 3
__global__ void refine_accum_kernel(const double* __restrict__ Z, int64_t n, int first, double* __restrict__ x) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double v = Z[i] * (1.0 / 3.0);
  x[i] = first ? v : x[i] + v;
}

// ---------------------------------------------------------------- soft inverse by a Chebyshev expansion
// With G = T + sigma I = L L^T and P = L^-1 (rocSOLVER's lower triangle, i.e.
// row r of the row-major n x n array holds P_{c r} at columns c >= r), M =
// T G^-1 = I - sigma P^T P is symmetric with the eigenvectors of T and
// eigenvalues mu = v / (v + sigma) in [0, mu_max]; g(T) = h(M) with h(mu) =
// g(sigma mu / (1 - mu)), a function analytic on [0, mu_max] whose nearest
// poles (from those of g at v = c e^{i pi (2k+1)/6}) stay ~0.13 away for
// sigma = c, so its Chebyshev series converges by ~1.3 per term.  Each term
// costs one P product and one P^T product, both half-row streams of the
// array once the strictly lower part (row-major) holds the transpose of the
// upper one.

// S[r n + c] = S[c n + r] for c < r: 64 x 64 tiles through LDS (rows padded
// to 65 doubles against bank conflicts); one workgroup per lower tile
__global__ __launch_bounds__(256) void tri_mirror_kernel(double* __restrict__ S, int64_t n, int nt) {
  __shared__ double buf[64][65];
  // lower tile (tr, tc), tr >= tc, from the linear index
  int64_t q = blockIdx.x;
  int tr = (int)((sqrt(8.0 * (double)q + 1.0) - 1.0) * 0.5);
  while ((int64_t)(tr + 1) * (tr + 2) / 2 <= q) ++tr;
  while ((int64_t)tr * (tr + 1) / 2 > q) --tr;
  const int tc = (int)(q - (int64_t)tr * (tr + 1) / 2);
  if (tr >= nt) return;
  const int64_t r0 = (int64_t)tr * 64, c0 = (int64_t)tc * 64;
  const int tx = threadIdx.x % 64, ty = threadIdx.x / 64;
  // source tile: rows c0.., columns r0.. (the upper part)
  for (int a = ty; a < 64; a += 4) {
    const int64_t sr = c0 + a, sc = r0 + tx;
    buf[a][tx] = (sr < n && sc < n) ? S[sr * n + sc] : 0.0;
  }
  __syncthreads();
  for (int b = ty; b < 64; b += 4) {
    const int64_t r = r0 + b, c = c0 + tx;
    if (r < n && c < n && c < r) S[r * n + c] = buf[tx][b];
  }
}

// Y = P X (LOWER: row i, columns c <= i) or P^T X (upper: columns c >= i):
// one wave per row, coalesced reads along the row
template <bool LOWER>
__global__ __launch_bounds__(256) void tri_rows_kernel(const double* __restrict__ S, int64_t n,
                                                       const double* __restrict__ X, double* __restrict__ Y) {
  const int lane = threadIdx.x % WAVE;
  const int64_t i = (int64_t)blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE;
  if (i >= n) return;
  const double* row = S + i * n;
  const double acc = wave_sum(wave_row_dot(row, X, LOWER ? 0 : i, LOWER ? i + 1 : n, lane));
  if (lane == 0) Y[i] = acc;
}

// One Chebyshev term: w = P^T u (upper half rows) fused with the recurrence
// t_{k+1} = 2 (alpha t_k - beta w) - t_{k-1} (first: t_1 = alpha t_0 - beta w,
// x = a0 t_0 + a t_1), x += a t_{k+1}; A = alpha I - beta P^T P maps the
// spectrum of M onto [-1, 1].  t_{k+1} replaces t_{k-1} in tprev.
__global__ __launch_bounds__(256) void cheb_rows_kernel(const double* __restrict__ S, int64_t n,
                                                        const double* __restrict__ u, const double* __restrict__ tcur,
                                                        double* __restrict__ tprev, double alpha, double beta,
                                                        double a0, double a, int first, double* __restrict__ x) {
  const int lane = threadIdx.x % WAVE;
  const int64_t i = (int64_t)blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE;
  if (i >= n) return;
  const double w = wave_sum(wave_row_dot(S + i * n, u, i, n, lane));
  if (lane == 0) {
    const double tk = tcur[i];
    const double tn = first ? alpha * tk - beta * w : 2.0 * (alpha * tk - beta * w) - tprev[i];
    tprev[i] = tn;
    x[i] = first ? a0 * tk + a * tn : x[i] + a * tn;
  }
}

// p: 2 H values per lane, summed over lane pairs S H apart; lanes with that bit
// set keep the upper half of the values
template <int H, int S>
__device__ __forceinline__ void halve_columns(double* p, int lane) {
  const bool up = lane & (S * H);
#pragma unroll
  for (int i = 0; i < H; ++i) {
    const double keep = up ? p[i + H] : p[i], send = up ? p[i] : p[i + H];
    p[i] = keep + __shfl_xor(send, S * H, WAVE);
  }
}

// One read of a triangle for both of its products (n <= kTriPassMax).  A
// workgroup of 512 threads (one per CU) takes rows c of the lower triangle
// (row-major, columns j <= c), RB at a time: a thread holds the rows' columns
// 2 t + 1024 i in registers, x is in LDS, the next rows are in flight while
// these are used, and the row's multiples are added to the workgroup's partial
// result in registers.
//   SYM = false: w = P^T (P x): u_c = row . x, w += u_c row (one barrier a turn
//                for the sum over the workgroup)
//   SYM = true:  y = T x for symmetric T: y_c += row . x (columns j < c; the
//                sums over the workgroup are taken once, at the end), y += x_c row
// part: (gridDim.x, n) partial results; dots: n (SYM).  HBM-bound: half the
// bytes of two half-row passes (P) or of full rows (T).
constexpr int TP_THREADS = 512, TP_WAVES = TP_THREADS / WAVE;
constexpr int TP_GRID = 256;  // one workgroup per CU (x fills most of the LDS)
// Where one read of half the matrix wins.  Below, the matrix comes from the
// last-level cache and the partial results cost more than the second read
// (us, two reads | one and its sum):
//   n      T x          P^T P x
//   2560    9.8 | 16.4   17.2 | 16.9
//   3072   12.2 | 17.6   21.1 | 17.9
//   4096   21.6 | 21.7   30.2 | 22.6
//   5000   34.2 | 30.6   41.8 | 33.1
//   8192   84.5 | 56.8   98.7 | 60.3
//   16384   329 |  216    360 |  223  (1.07 GB: 5.0 TB/s)
constexpr int64_t kTriPassSymMin = 4608, kTriPassMin = 2560, kTriPassMax = 16384;
typedef double v2d_u __attribute__((ext_vector_type(2), aligned(8)));

template <int NC>
constexpr int tp_lds() {  // x, then the waves' sums of every row (at most kTriPassMax / TP_GRID turns of one row)
  return 2 * TP_THREADS * NC * 8 + (int)(kTriPassMax / TP_GRID) * TP_WAVES * 8;
}

template <int RB, int NC, bool SYM>
__global__ __launch_bounds__(TP_THREADS) void tri_pass_kernel(const double* __restrict__ S, int64_t n,
                                                              const double* __restrict__ X,
                                                              double* __restrict__ part, double* __restrict__ dots) {
  static_assert(RB * TP_WAVES <= WAVE, "one lane per wave's sum");
  extern __shared__ __attribute__((aligned(16))) double tp[];
  double* xs = tp;                         // 2 TP_THREADS NC, zero past n
  double* red = tp + 2 * TP_THREADS * NC;  // [turn (SYM) or turn % 2][RB][TP_WAVES]
  const int t = threadIdx.x, lane = t % WAVE, wv = t / WAVE;
  for (int j = t; j < 2 * TP_THREADS * NC; j += TP_THREADS) xs[j] = j < n ? X[j] : 0.0;
  __syncthreads();
  v2d_u w[NC], row[2][RB][NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) w[i] = v2d_u{0.0, 0.0};
  auto row_of = [&](int turn, int r) { return ((int64_t)turn * TP_GRID + blockIdx.x) * RB + r; };
  auto load = [&](int turn, v2d_u (&b)[RB][NC]) {
    int off = 16 * t;
    asm volatile("" : "+v"(off));  // the NC offsets are formed in every turn, not kept in registers
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int64_t c = row_of(turn, r);
      // the row up to its diagonal; columns past it (and rows past n) read as zero
      const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)(S + (c < n ? c * n : 0)), 0,
                                                        c < n ? (int)(c + 1) * 8 : 0, 0x00020000);
#pragma unroll
      for (int i = 0; i < NC; ++i)
        b[r][i] = __builtin_bit_cast(v2d_u, __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16 * TP_THREADS * i, 0, 0));
    }
  };
  auto use = [&](int turn, v2d_u (&b)[RB][NC]) {
    asm volatile("" ::: "memory");  // x is read from LDS in every turn, not kept in registers
    double* rd = red + (SYM ? turn : (turn & 1)) * RB * TP_WAVES;
    double p[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      int d = 2 * t - (int)row_of(turn, r);  // the diagonal is at column 2 t - d
      asm volatile("" : "+v"(d));
      p[r] = 0.0;
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        if (NC > 4 && i % 4 == 0) __builtin_amdgcn_sched_barrier(0);  // few of x's reads at a time
        const double2 x2 = *reinterpret_cast<const double2*>(xs + 2 * t + 2 * TP_THREADS * i);
        if (d == -2 * TP_THREADS * i) b[r][i].y = 0.0;  // the second of the last pair, if there is one to read
        // the diagonal of T belongs to the row's multiple
        p[r] += (SYM && d == -2 * TP_THREADS * i ? 0.0 : b[r][i].x) * x2.x +
                (SYM && d == -2 * TP_THREADS * i - 1 ? 0.0 : b[r][i].y) * x2.y;
      }
    }
    // the RB sums of a wave by one butterfly; row r ends in the r-th WAVE / RB lanes
    if constexpr (RB == 4) halve_columns<2, 16>(p, lane);
    if constexpr (RB >= 2) halve_columns<1, RB == 4 ? 16 : 32>(p, lane);
    for (int q = WAVE / RB / 2; q >= 1; q /= 2) p[0] += __shfl_xor(p[0], q, WAVE);
    if (lane % (WAVE / RB) == 0) rd[lane / (WAVE / RB) * TP_WAVES + wv] = p[0];
    double sums = 0.0;
    if (!SYM) {
      __syncthreads();
      sums = rd[lane % (RB * TP_WAVES)];
      for (int q = 1; q < TP_WAVES; q *= 2) sums += __shfl_xor(sums, q, WAVE);
    }
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int64_t c = row_of(turn, r);
      const double u = SYM ? (c < n ? xs[c] : 0.0) : readlane_f64(sums, r * TP_WAVES);
#pragma unroll
      for (int i = 0; i < NC; ++i) w[i] += u * b[r][i];
    }
  };
  const int turns = (int)((n + (int64_t)TP_GRID * RB - 1) / ((int64_t)TP_GRID * RB));
  load(0, row[0]);
  for (int k = 0; k < turns; k += 2) {  // a turn past the last loads nothing: its rows are past n
    load(k + 1, row[1]);
    use(k, row[0]);
    if (k + 1 == turns) break;
    load(k + 2, row[0]);
    use(k + 1, row[1]);
  }
  double* out = part + (int64_t)blockIdx.x * n;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int64_t j = 2 * t + 2 * TP_THREADS * i;
    if (j < n) out[j] = w[i].x;
    if (j + 1 < n) out[j + 1] = w[i].y;
  }
  if (SYM) {
    __syncthreads();
    for (int e = t; e < turns * RB; e += TP_THREADS) {
      const int64_t c = row_of(e / RB, e % RB);
      if (c < n) {
        double u = 0.0;
#pragma unroll
        for (int q = 0; q < TP_WAVES; ++q) u += red[e * TP_WAVES + q];
        dots[c] = u;
      }
    }
  }
}

// sums over the TP_GRID partial results of TP_COLS columns, for threads t < TP_COLS
constexpr int TP_COLS = 16;
__device__ __forceinline__ double tp_column_sum(const double* __restrict__ part, int64_t n, int64_t j) {
  __shared__ double sh[1024 / WAVE][TP_COLS];
  const int t = threadIdx.x, grp = t / TP_COLS;
  double a = 0.0;
  if (j < n) {
    double v[TP_GRID * TP_COLS / 1024];
#pragma unroll
    for (int k = 0; k < TP_GRID * TP_COLS / 1024; ++k) v[k] = part[(int64_t)(grp + k * (1024 / TP_COLS)) * n + j];
#pragma unroll
    for (int k = 0; k < TP_GRID * TP_COLS / 1024; ++k) a += v[k];
  }
  a += __shfl_xor(a, 16, WAVE);
  a += __shfl_xor(a, 32, WAVE);
  if (t % WAVE < TP_COLS) sh[t / WAVE][t % WAVE] = a;
  __syncthreads();
  double s = 0.0;
  if (t < TP_COLS)
#pragma unroll
    for (int q = 0; q < 1024 / WAVE; ++q) s += sh[q][t];
  return s;
}

// y = T x from tri_pass_kernel<SYM>
__global__ __launch_bounds__(1024) void tp_sum_kernel(const double* __restrict__ part, const double* __restrict__ dots,
                                                      int64_t n, double* __restrict__ y) {
  const int64_t j = (int64_t)blockIdx.x * TP_COLS + threadIdx.x % TP_COLS;
  const double s = tp_column_sum(part, n, j);
  if (threadIdx.x < TP_COLS && j < n) y[j] = s + dots[j];
}

// the Chebyshev recurrence of cheb_rows_kernel on w = P^T P t_k from tri_pass_kernel
__global__ __launch_bounds__(1024) void tp_cheb_kernel(const double* __restrict__ part, int64_t n,
                                                       const double* __restrict__ tcur, double* __restrict__ tprev,
                                                       double alpha, double beta, double a0, double a, int first,
                                                       double* __restrict__ x) {
  const int64_t i = (int64_t)blockIdx.x * TP_COLS + threadIdx.x % TP_COLS;
  const double w = tp_column_sum(part, n, i);
  if (threadIdx.x < TP_COLS && i < n) {
    const double tk = tcur[i];
    const double tn = first ? alpha * tk - beta * w : 2.0 * (alpha * tk - beta * w) - tprev[i];
    tprev[i] = tn;
    x[i] = first ? a0 * tk + a * tn : x[i] + a * tn;
  }
}

// single block: out[0] = |a|^2, out[1] = |b|^2
__global__ __launch_bounds__(1024) void sq_norms_kernel(const double* __restrict__ a, const double* __restrict__ b,
                                                        int64_t n, double* __restrict__ out) {
  __shared__ double red[16];
  double sa = 0.0, sb = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    sa += a[i] * a[i];
    sb += b[i] * b[i];
  }
  sa = block_sum_1024(sa, red);
  sb = block_sum_1024(sb, red);
  if (threadIdx.x == 0) {
    out[0] = sa;
    out[1] = sb;
  }
}

// ---------------------------------------------------------------- SNR truncation
// _sum_without_noise (optimizer/solver.py:114-125): rho_s = sum_t c_ts is
// divided by 1 + (tol / snr_s)^6, snr_s = |mean_s| / sqrt(var_s / m), with the
// variance about the mean as the reference forms it (two passes: rho is known
// before the sums of squares are taken).
// var2[s] = sum_t (U[t, s] y[t] - rho[s] / m)^2, U column-major n x n, one
// block per column (MinSR and minsr_pinv_eig: c_ts = U_ts b_t)
__global__ __launch_bounds__(256) void snr_colsq_kernel(const double* __restrict__ U, int64_t n,
                                                        const double* __restrict__ y, const double* __restrict__ rho,
                                                        double m, double* __restrict__ var2) {
  __shared__ double red[4];
  const int64_t s = blockIdx.x;
  const double* col = U + s * n;
  const double mu = rho[s] / m;
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    const double v = col[i] * y[i] - mu;
    acc += v * v;
  }
  acc = wave_sum(acc);
  if (threadIdx.x % WAVE == 0) red[threadIdx.x / WAVE] = acc;
  __syncthreads();
  if (threadIdx.x == 0) var2[s] = red[0] + red[1] + red[2] + red[3];
}

// var2[k] (+)= sum_s (C[k + s np] e[s] - rho[k] / m)^2 over a block of rows s
// (C = Obar V of the block, column-major np x rows: SR, c_sk = (Obar V)_sk Ebar_s)
__global__ __launch_bounds__(256) void snr_rowsq_kernel(const double* __restrict__ Cb, int64_t np, int64_t rows,
                                                        const double* __restrict__ e, const double* __restrict__ rho,
                                                        double m, int first, double* __restrict__ var2) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= np) return;
  const double mu = rho[k] / m;
  double acc = 0.0;
  for (int64_t s = 0; s < rows; ++s) {
    const double v = Cb[k + s * np] * e[s] - mu;
    acc += v * v;
  }
  var2[k] = (first ? 0.0 : var2[k]) + acc;
}

__global__ void snr_scale_kernel(double* __restrict__ rho, const double* __restrict__ var2, int64_t n, double m,
                                 double tol) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  // rho = 0 stays 0 (the reference's 0 / (1 + (tol / (0/0))^6) is NaN there)
  if (rho[i] == 0.0) return;
  const double mean = rho[i] / m;
  const double snr = fabs(mean) / sqrt(var2[i] / m / m);
  const double q = tol / snr, q2 = q * q;
  rho[i] = rho[i] / (1.0 + q2 * q2 * q2);
}

// ---------------------------------------------------------------- rocBLAS handle
// One handle per (thread, device, stream).  A handle carries the device
// workspace rocSOLVER uses for its temporaries, so one handle switched between
// streams would let two factorisations in flight on different streams share
// that scratch; a handle bound to a single stream cannot.  Two caches: handles
// whose scratch rocBLAS allocates and keeps (the default), and handles that
// only ever use scratch the caller brings in its workspace (QTX_SOLVE_BLAS_WS:
// rocblas_set_workspace before every use, so rocBLAS allocates nothing).  Each
// keeps at most kMaxHandles per thread and device; the oldest is retired after
// a device-wide sync.
constexpr size_t kMaxHandles = 64;
struct BlasEntry {
  hipStream_t stream;
  rocblas_handle handle;
};
static thread_local std::vector<BlasEntry> g_blas[64];
static thread_local std::vector<BlasEntry> g_blas_user[64];

static int get_blas(hipStream_t st, rocblas_handle* h, void* user_ws = nullptr, size_t user_bytes = 0,
                    bool user = false) {
  int dev = 0;
  QTX_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return fail(QTX_EHIP, "device index out of range");
  std::vector<BlasEntry>& cache = user ? g_blas_user[dev] : g_blas[dev];
  rocblas_handle found = nullptr;
  for (const BlasEntry& e : cache)
    if (e.stream == st) found = e.handle;
  if (!found) {
    if (cache.size() >= kMaxHandles) {
      QTX_HIP(hipDeviceSynchronize());
      rocblas_destroy_handle(cache.front().handle);
      cache.erase(cache.begin());
    }
    if (rocblas_create_handle(&found) != rocblas_status_success)
      return fail(QTX_ESOLVER, "rocblas_create_handle failed");
    if (rocblas_set_stream(found, st) != rocblas_status_success) {
      rocblas_destroy_handle(found);
      return fail(QTX_ESOLVER, "rocblas_set_stream failed");
    }
    cache.push_back(BlasEntry{st, found});
  }
  if (user && rocblas_set_workspace(found, user_ws, user_bytes) != rocblas_status_success)
    return fail(QTX_ESOLVER, "rocblas_set_workspace failed");
  *h = found;
  return QTX_OK;
}

static int rb(rocblas_status s, const char* what) {
  if (s == rocblas_status_success) return QTX_OK;
  if (s == rocblas_status_memory_error)
    return fail(QTX_EWORKSPACE, std::string(what) + ": rocBLAS/rocSOLVER scratch does not fit (with "
                                "QTX_SOLVE_BLAS_WS, size the workspace tail by qtx_minsr_blas_ws_bytes)");
  return fail(QTX_ESOLVER, std::string(what) + " failed: " + rocblas_status_to_string(s));
}

}  // namespace qtx

using namespace qtx;

static int nblk(int64_t n, int b) { return (int)((n + b - 1) / b); }
// grid cap of the grid-stride element-wise kernels (256-thread blocks): the
// work-item count of one launch must stay below 2^32
constexpr int64_t kGridCap = int64_t(1) << 20;

constexpr int kLanczosMax = 512;  // Lanczos steps for lambda_max before giving up on convergence
#ifndef QTX_CHOL_BLOCK
#define QTX_CHOL_BLOCK 1024
#endif
constexpr int64_t kCholBlock = QTX_CHOL_BLOCK;  // diagonal block of the blocked Cholesky
// Width of the diagonal block that starts with `rem` columns left: the rest of the
// matrix once the panel and update kernels do it faster than dtrsm and dsyrk on
// its blocks (the rank-64 updates then come from the last-level cache): 4096 3.85
// -> 2.99 ms, 6144 7.7 -> 6.4, the last 6144 of 12288 31.0 -> 29.7, of 16384 58.6
// -> 57.5 (8192: 58.4); three matrices of 2000 7.0 -> 5.35 ms for their solve.
static int64_t chol_block(int64_t rem, int batch) {
  return rem <= (batch == 1 ? 6144 : 2048) ? rem : kCholBlock;
}
constexpr int kInfoPerFactor = (int)((131072 + kCholBlock - 1) / kCholBlock);  // status slots: n <= 131072

// Rows of FP64 Obar formed per DGEMM chunk in the SR branch (<= 256 MiB)
static int64_t obar_rows(int64_t ns, int64_t np) {
  return std::max<int64_t>(1, std::min<int64_t>(ns, (int64_t(1) << 28) / (8 * std::max<int64_t>(np, 1))));
}

// solver mode without its flags, and the branch: T = Obar Obar^T (MinSR) or
// S = Obar^T Obar (SR), by the flags or, without them, by the shape
static inline int base_mode(int mode) { return mode & 0xff; }
static inline bool use_minnorm(int64_t ns, int64_t np, int mode) {
  if (mode & QTX_SOLVE_MINNORM) return true;
  if (mode & QTX_SOLVE_LSTSQ) return false;
  return ns < np;
}
constexpr double kSnrMin = 1e-6;  // tol_snr at or below it: no truncation (solver.py:124)
// Chebyshev route (cutoffs c >= 1e-5 lambda_max): taken from n >= kChebMinN
// on, where its one factorisation and triangular inverse plus ~2 n^2 x 8 B
// of streaming per term cost less than the partial fractions' T^2 and three
// factorisations (measured: 6.4 against 7.1 ms at n = 2048, 15 against 18 ms
// at 4096, 2.4 against 2.0 ms at 512), or whenever QTX_SOLVE_CHEB asks for
// it.  Terms up to kChebMax; the series is cut where 8 consecutive
// coefficients fall below kChebTol of the largest (about 158 terms).
constexpr int64_t kChebMinN = 2048;
constexpr int kChebMax = 400;
constexpr int kChebNodes = 1024;
constexpr double kChebTol = 1e-15;
// The series covers mu down to -kChebMargin (eigenvalues of T down to -c / 6,
// which rounding in the split-bf16 Gram can produce), and the last term's norm
// is checked against the right-hand side's: a Chebyshev polynomial is bounded
// by 1 on the interval, so growth means T has eigenvalues below it, and the
// solve takes the partial fractions instead.
constexpr double kChebMargin = 0.2;
constexpr double kChebGrowth = 1.5;
// shifted Cholesky route: G = T_d - kShiftCut c I must factor, which puts every
// eigenvalue of T_d above 150 c, where the soft inverse differs from 1/v by
// (c/v)^6 <= 8.8e-14; kShiftIters preconditioned CG steps, accepted when the
// true residual's normwise backward error |b' - T_d x| / (lambda_max |x|) is
// below kShiftAccept (the accuracy a backward-stable eigensolver attains)
constexpr double kShiftCut = 150.0;
constexpr int kShiftIters = 40;
constexpr double kShiftAccept = 1e-15;

struct SolveWs {
  double* T;       // n x n
  double* y;       // max(ns, np)
  double* z;       // max(ns, np)
  double* D;       // n
  double* E;       // n
  double* scalars; // 8: trace, power-of-two scale, whether the weights are one (MinSR), -, four norms
  int32_t* info;   // 4 (+pad)
  double* dtile;   // 3 x 64 x 64: factored diagonal tiles of the blocked Cholesky, staged
  // partial-fraction soft inverse (EIGH_PINV modes only)
  double* T2;      // 3 x (n x n): T^2 (lower), then the three (T - a_k)^2 + b_k^2
                   // (the first in place of T^2) and their Cholesky factors
  double* R;       // n x 6: residuals, then A_k^{-1} residuals (pole k: columns 2k, 2k+1)
  double* TW;      // n x 6: T times those vectors
  double* Z;       // n x 2: complex solution
  double* x;       // n: accumulated soft-inverse solution
  double* V;       // 3n: Lanczos vectors
  double* w;       // n: Lanczos work vector
  double* ab;      // alpha[kLanczosMax], beta[kLanczosMax + 1]
  void* split;     // bf16 hi / lo planes of Obar (split-bf16 Gram only)
  double* obar;    // obar_rows x np FP64 Obar of a row block (SR branch, where needs_obar)
  double* var2;    // n: SNR truncation, sums of squared deviations (QTX_SOLVE_SNR)
  double* cbuf;    // obar_rows x np: Obar V of a row block (SR branch with QTX_SOLVE_SNR)
};

static size_t ws_layout(int64_t ns, int64_t np, int mode, int gram, SolveWs* w, char* base) {
  const bool mn = use_minnorm(ns, np, mode);
  int64_t n = mn ? ns : np;
  int64_t m = ns > np ? ns : np;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    size_t o = off;
    off += (bytes + 255) & ~(size_t)255;
    return base ? base + o : nullptr;
  };
  SolveWs s{};
  s.T = (double*)take((size_t)n * n * 8);
  s.y = (double*)take((size_t)m * 8);
  s.z = (double*)take((size_t)m * 8);
  s.D = (double*)take((size_t)n * 8);
  s.E = (double*)take((size_t)n * 8);
  s.scalars = (double*)take(64);
  s.info = (int32_t*)take(3 * kInfoPerFactor * sizeof(int32_t));
  s.dtile = (double*)take((size_t)3 * 64 * 64 * 8);
  if (base_mode(mode) == QTX_SOLVE_EIGH_PINV) {
    s.T2 = (double*)take((size_t)3 * n * n * 8);
    s.R = (double*)take((size_t)n * 48);
    s.TW = (double*)take((size_t)n * 48);
    s.Z = (double*)take((size_t)n * 48);
    s.x = (double*)take((size_t)n * 8);
    s.V = (double*)take((size_t)n * 24);
    s.w = (double*)take((size_t)n * 8);
    s.ab = (double*)take((size_t)(2 * kLanczosMax + 1) * 8);
  }
  if (gram == QTX_GRAM_BF16X3 && mn) s.split = take(g3_bytes(ns, np));
  if (!mn && needs_obar(np, mode)) s.obar = (double*)take((size_t)obar_rows(ns, np) * np * 8);
  if (mode & QTX_SOLVE_SNR) {
    s.var2 = (double*)take((size_t)n * 8);
    if (!mn) s.cbuf = (double*)take((size_t)obar_rows(ns, np) * np * 8);
  }
  if (w) *w = s;
  return off;
}

// what the last qtx_minsr_solve on this thread did
static thread_local int g_last_path = -1;
static thread_local int g_last_lanczos = 0;
static thread_local double g_last_lmax = 0.0;
static thread_local int g_last_fallback = 0;  // why the partial-fraction route was left (0: it was not)

// largest eigenvalue of the m x m symmetric tridiagonal (diag a[0..m), off-diagonal
// e[1..m) between rows i-1 and i) by Sturm-count bisection
static double tridiag_max_eig(const double* a, const double* e, int m) {
  double lo = a[0], hi = a[0];
  for (int i = 0; i < m; ++i) {
    double r = (i > 0 ? fabs(e[i]) : 0.0) + (i + 1 < m ? fabs(e[i + 1]) : 0.0);
    lo = fmin(lo, a[i] - r);
    hi = fmax(hi, a[i] + r);
  }
  auto count_below = [&](double x) {
    int c = 0;
    double q = a[0] - x;
    for (int i = 0;;) {
      if (q == 0.0) q = -1e-300;
      if (q < 0.0) ++c;
      if (++i >= m) break;
      q = a[i] - x - e[i] * e[i] / q;
    }
    return c;
  };
  for (int it = 0; it < 256 && hi - lo > 2e-16 * fmax(fabs(lo), fabs(hi)); ++it) {
    double mid = 0.5 * (lo + hi);
    if (mid <= lo || mid >= hi) break;
    if (count_below(mid) == m) hi = mid;
    else lo = mid;
  }
  return hi;
}

template <typename TI>
static int launch_gram_nt(hipStream_t st, int gram, const TI* O, const double* mean, const double* r, int64_t n,
                          int64_t np, double* T, void* split_ws) {
  int64_t nt = (n + GT - 1) / GT;
  int64_t ntiles = nt * (nt + 1) / 2;
  QTX_REQUIRE(ntiles < 0x7fffffff, "Gram too large");
  dim3 g((unsigned)ntiles), bl(256);
  double inv_ns = 1.0 / (double)n;
  if (gram == QTX_GRAM_BF16X3) {
    QTX_REQUIRE(split_ws != nullptr, "split-bf16 Gram needs its workspace");
    const int64_t rows = g3_rows(n), kpad = g3_kpad(np), bpr = (kpad + 256 * SP_COLS - 1) / (256 * SP_COLS);
    const int64_t nblocks = rows * bpr;
    __bf16* HL = (__bf16*)split_ws;
    hipLaunchKernelGGL(split_bf16x3_kernel<TI>, dim3((unsigned)std::min<int64_t>(nblocks, kGridCap)), dim3(256), 0,
                       st, O, mean, r, n, np, kpad, bpr, nblocks, inv_ns, HL);
    if (nt >= G3_DEAL) {
      const int64_t ms = (nt + 7) / 8, sb = ms * (ms + 1) / 2;
      QTX_REQUIRE((sb + 7) / 8 * 512 < 0x7fffffff, "Gram too large");
      g = dim3((unsigned)((sb + 7) / 8 * 512));
    }
    hipLaunchKernelGGL(gram_bf16x3_kernel, g, bl, 0, st, (const __bf16*)HL, n, kpad, (int)ntiles, T);
  } else {
    const int64_t mt = (n + GN_T - 1) / GN_T, mtiles = mt * (mt + 1) / 2;
    QTX_REQUIRE(mtiles < 0x7fffffff, "Gram too large");
    const int64_t per = (mtiles + 7) / 8, whole = gram_whole((int)per);
    const dim3 gm((unsigned)(8 * (whole + 4 * (per - whole))));
    if (gram == QTX_GRAM_FP32)
      hipLaunchKernelGGL((gram_nt_kernel<TI, QTX_GRAM_FP32>), gm, bl, 0, st, O, mean, r, n, np, inv_ns, (int)mtiles, T);
    else
      hipLaunchKernelGGL((gram_nt_kernel<TI, QTX_GRAM_FP64>), gm, bl, 0, st, O, mean, r, n, np, inv_ns, (int)mtiles, T);
  }
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

template <typename TI>
static int launch_obar_t_y(hipStream_t st, const TI* O, const double* mean, const double* r, const double* y,
                           int64_t ns, int64_t np, double* x) {
  hipLaunchKernelGGL(fill_f64_kernel, dim3(nblk(np, 256)), dim3(256), 0, st, x, np, 0.0);
  dim3 g;
  int lg;
  const int64_t rpc = colsum_rows(ns, np, g, lg);
  hipLaunchKernelGGL((colsum_kernel<TI, true>), g, dim3(256), 0, st, O, mean, r, y, ns, np, rpc, lg, 1.0 / (double)ns,
                     x);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

// What the SNR truncation of the SR branch needs besides the eigenvectors:
// the per-sample contributions are (Obar V)_sk Ebar_s, Obar formed again a
// row block at a time
struct SnrRows {
  int o_dtype;
  const void* O;
  const double* mean;
  const double* r;
  const double* ebar;
  int64_t ns, np;
};

template <typename TI>
static int snr_rows_var2(hipStream_t st, rocblas_handle h, const SnrRows& L, SolveWs& w) {
  const int64_t rows = obar_rows(L.ns, L.np);
  const double one = 1.0, zero = 0.0;
  const TI* O = (const TI*)L.O;
  for (int64_t s0 = 0; s0 < L.ns; s0 += rows) {
    const int64_t nr = std::min(rows, L.ns - s0), tot = nr * L.np;
    hipLaunchKernelGGL(form_obar_kernel<TI>, dim3((unsigned)std::min<int64_t>((tot + 255) / 256, kGridCap)), dim3(256),
                       0, st, O + s0 * L.np, L.mean, L.r ? L.r + s0 : nullptr, nr, L.np, 1.0 / (double)L.ns, w.obar);
    QTX_LAUNCH_CHECK();
    // (Obar V)^T of the block, column-major np x nr: V^T B with B the block
    // as a column-major np x nr matrix
    int rc = rb(rocblas_dgemm(h, rocblas_operation_transpose, rocblas_operation_none, (rocblas_int)L.np,
                              (rocblas_int)nr, (rocblas_int)L.np, &one, w.T, (rocblas_int)L.np, w.obar,
                              (rocblas_int)L.np, &zero, w.cbuf, (rocblas_int)L.np),
                "rocblas_dgemm");
    if (rc) return rc;
    hipLaunchKernelGGL(snr_rowsq_kernel, dim3(nblk(L.np, 256)), dim3(256), 0, st, w.cbuf, L.np, nr, L.ebar + s0, w.z,
                       (double)L.ns, s0 == 0 ? 1 : 0, w.var2);
    QTX_LAUNCH_CHECK();
  }
  return QTX_OK;
}

// y <- U g(D) U^T y through rocSOLVER dsyevd (T is overwritten); with
// tol_snr > 1e-6 the components of U^T y are truncated by their SNR (rows ==
// nullptr: c_ts = U_ts y_t over the n rows of T; else the SR branch's
// (Obar V)_sk Ebar_s over the samples); returns 1 or an error
static int pinv_syevd(hipStream_t st, rocblas_handle h, int64_t n, double rtol, double atol, SolveWs& w,
                      double tol_snr = 0.0, const SnrRows* rows = nullptr) {
  const rocblas_int ni = (rocblas_int)n;
  // exact power-of-two rescaling of T (eigenvectors unchanged, eigenvalues
  // scaled by 2^k and undone in eig_inv_kernel)
  hipLaunchKernelGGL(pow2_scale_kernel, dim3(1), dim3(1024), 0, st, w.T, n, w.scalars + 1);
  hipLaunchKernelGGL(scale_by_kernel, dim3((unsigned)std::min<int64_t>((n * n + 255) / 256, kGridCap)), dim3(256), 0,
                     st, w.T, n * n,
                     w.scalars + 1);
  QTX_LAUNCH_CHECK();
  int rc = rb(rocsolver_dsyevd(h, rocblas_evect_original, rocblas_fill_lower, ni, w.T, ni, w.D, w.E, w.info),
              "rocsolver_dsyevd");
  if (rc) return rc;
  const double one = 1.0, zero = 0.0;
  // z = U^T y ; z *= eig_inv ; y = U z   (U column-major in T)
  rc = rb(rocblas_dgemv(h, rocblas_operation_transpose, ni, ni, &one, w.T, ni, w.y, 1, &zero, w.z, 1),
          "rocblas_dgemv");
  if (rc) return rc;
  if (tol_snr > kSnrMin) {
    QTX_REQUIRE(w.var2 != nullptr, "tol_snr > 0 needs the QTX_SOLVE_SNR workspace");
    double m = (double)n;
    if (rows == nullptr) {
      hipLaunchKernelGGL(snr_colsq_kernel, dim3((unsigned)n), dim3(256), 0, st, w.T, n, w.y, w.z, m, w.var2);
      QTX_LAUNCH_CHECK();
    } else {
      QTX_REQUIRE(w.cbuf != nullptr, "tol_snr > 0 needs the QTX_SOLVE_SNR workspace");
      rc = rows->o_dtype == QTX_F32 ? snr_rows_var2<float>(st, h, *rows, w) : snr_rows_var2<double>(st, h, *rows, w);
      if (rc) return rc;
      m = (double)rows->ns;
    }
    hipLaunchKernelGGL(snr_scale_kernel, dim3(nblk(n, 256)), dim3(256), 0, st, w.z, w.var2, n, m, tol_snr);
    QTX_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(eig_inv_kernel, dim3(1), dim3(1024), 0, st, w.D, n, rtol, atol, w.scalars + 1, w.z);
  QTX_LAUNCH_CHECK();
  rc = rb(rocblas_dgemv(h, rocblas_operation_none, ni, ni, &one, w.T, ni, w.z, 1, &zero, w.y, 1), "rocblas_dgemv");
  if (rc) return rc;
  int32_t info_h = 0;
  QTX_HIP(hipMemcpyAsync(&info_h, w.info, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  QTX_HIP(hipStreamSynchronize(st));
  if (info_h != 0) return fail(QTX_ESOLVER, "syevd info = " + std::to_string(info_h));
  g_last_path = 2;
  return 1;
}

// ---------------------------------------------------------------- Cholesky
// Right-looking blocked Cholesky (lower, column-major, leading dimension n) of
// `batch` matrices `stride` elements apart.  Each diagonal block (kCholBlock
// columns, or all that is left: chol_block) is factored in CT-column panels by two kernels of this file (panel:
// factor the CT x CT diagonal tile in LDS and solve the tiles below it inside
// the block; update: the rank-CT update of the block's remaining tiles), all
// matrices in one launch, so the latency-bound diagonal work of one matrix
// overlaps that of the others; the rows below a diagonal block are then solved
// by rocBLAS dtrsm and the trailing matrix updated by dsyrk, matrix by matrix,
// so nearly all flops run in level-3 BLAS kernels.  info[b * info_stride + blk]
// receives 1 + the column (within diagonal block blk) of the first
// non-positive pivot of matrix b, 0 if none; as in LAPACK, that matrix's
// factor is not usable then (NaNs propagate, the other matrices are
// unaffected).
constexpr int CT = 64;
constexpr int CL = 80;       // LDS stride of a tile's columns: the four columns of a fragment fall on distinct banks
constexpr int CI = 18;       // LDS stride of the columns of an inverted 16 x 16 block

// 1 / sqrt(d), d > 0: the hardware's estimate (relative error < 2^-23) and one
// third-order step; four dependent operations instead of a division after a
// square root, which every column of a factorisation waits for
__device__ __forceinline__ double rsqrt_f64(double d) {
  const double y = __builtin_amdgcn_rsq(d);
  const double e = __builtin_fma(-(d * y), y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
}

// base[off], 0 where !ok (base[0] is always readable): an address select instead
// of a branch around each load
__device__ __forceinline__ double load_or_zero(const double* base, int64_t off, bool ok) {
  const double v = base[ok ? off : 0];
  return ok ? v : 0.0;
}

// One panel: factor the 64 x 64 diagonal tile, then X = A_t L^-T for the tiles
// t below it inside the diagonal block.  Every workgroup factors the tile (it
// is a serial chain, so sharing it would cost a launch); workgroup 0 stores
// it, workgroup t solves tile t, the last one (with a right-hand side y) the
// 64 entries of y as one more row: y = L^-1 y when the factorisation ends.
//
// Bound by the chain of 64 pivots, and by the instruction fetch: nothing runs
// often, so a rolled loop is faster than a long unrolled one.  Wave q owns
// columns 16 q .. 16 q + 15.  A group of 8 columns is factored by its wave
// alone, one row per lane, with lane reads as broadcasts (no barrier inside a
// group); the columns after it then take the group's products by MFMA.  All
// MFMA work is on transposed tiles (D rows = columns of the matrix): D's
// element v of lane l is row 4 v + l / 16, which is also B's row of the K step
// v, so a solved block feeds the next products from its registers, and D's
// columns are matrix rows, contiguous in memory.
// The solve multiplies by the inverses of the four 16 x 16 diagonal blocks
// with one refinement against the block itself, which keeps the residual of
// substitution.  46 -> 18 us (one barrier, one division and one square root per
// column and register tiles before).
__global__ __launch_bounds__(256) void chol_panel_kernel(double* A, int64_t lda, int64_t stride, int64_t d0,
                                                         int64_t kb, int kp, int32_t* info, int64_t info_stride,
                                                         double* __restrict__ dtile, double* y) {
  __shared__ double Ls[CT * CL];
  __shared__ double Inv[4][16 * CI];
  __shared__ double rdg[CT];
  double* Ab = A + (int64_t)blockIdx.y * stride;
  const int tid = threadIdx.x, lane = tid % WAVE, g = lane / 16, m = lane % 16;
  const int q = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int64_t p0 = d0 + (int64_t)kp * CT;
  const int w = (int)(kb - (int64_t)kp * CT < CT ? kb - (int64_t)kp * CT : CT);
  const int nt = (int)((kb + CT - 1) / CT);
  const bool below = blockIdx.x > 0, yrow = (int)blockIdx.x == nt - kp;
  // this wave's 16 rows of the tile below (16 q ..), transposed: x[b][v] =
  // column 16 b + 4 v + g of row 16 q + m
  const int64_t q0 = p0 + (int64_t)blockIdx.x * CT;
  const int64_t hrem = kb - (int64_t)(kp + blockIdx.x) * CT;
  const int h = yrow ? 1 : (int)(hrem < CT ? hrem : CT);
  const double* Dp = Ab + p0 + p0 * lda;
  double* Xp = yrow ? y + p0 : Ab + q0 + p0 * lda;
  const int64_t xs = yrow ? 1 : lda;
  v4d c[4], x[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int col = 16 * q + 4 * v + g, row = 16 * b + m;
      c[b][v] = load_or_zero(Dp, row + col * lda, row < w && row >= col);
      if (row == col && row >= w) c[b][v] = 1.0;  // padding: identity
    }
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int xc = 16 * b + 4 * v + g, xr = 16 * q + m;
      x[b][v] = load_or_zero(Xp, xr + xc * xs, xr < h && xc < w);
    }
  int bad = -1;
  const int groups = (w + 7) / 8;  // a short last panel: the rest is the identity
  for (int c8 = 8 * groups + q; c8 < CT; c8 += 4) {
    Ls[c8 * CL + lane] = lane == c8 ? 1.0 : 0.0;
    rdg[c8] = 1.0;
  }
#pragma unroll 1
  for (int gb = 0; gb < groups; ++gb) {
    if (q == gb / 2) {
      // to one row per lane through these columns of Ls
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 2; ++v)
          Ls[(8 * gb + 4 * v + g) * CL + 16 * b + m] = (gb & 1) ? c[b][2 + v] : c[b][v];
      wave_lds_fence();
      double a[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) a[i] = Ls[(8 * gb + i) * CL + lane];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int row = 8 * gb + j;
        const double d = readlane_f64(a[j], row);
        if (!(d > 0.0) && bad < 0 && row < w) bad = row;  // NaN fails too
        const double rs = rsqrt_f64(d);
        a[j] *= rs;
#pragma unroll
        for (int i = j + 1; i < 8; ++i) a[i] -= a[j] * readlane_f64(a[j], 8 * gb + i);
        Ls[row * CL + lane] = lane >= row ? a[j] : 0.0;
        rdg[row] = rs;
      }
      if (blockIdx.x == 0 && lane == 0 && bad >= 0) {
        int32_t* slot = info + (int64_t)blockIdx.y * info_stride;
        if (*slot == 0) *slot = kp * CT + bad + 1;
      }
    }
    __syncthreads();
    if (2 * q + 1 > gb) {  // columns of this wave after the group (the ones before it are done with)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const double* lk = Ls + (8 * gb + 4 * s + g) * CL + m;
        const double lq = -lk[16 * q];
#pragma unroll
        for (int b = 0; b < 4; ++b) c[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(lq, lk[16 * b], c[b], 0, 0, 0);
      }
      mfma_settle_f64<4>(c);
    }
  }
  if (!below) {
    // staged, not stored into A: the other workgroups of this launch read the
    // unfactored tile from A, possibly after this one is done
    double* dt = dtile + (int64_t)blockIdx.y * CT * CT;
#pragma unroll
    for (int i = 0; i < 16; ++i) dt[(16 * q + i) * CT + lane] = Ls[(16 * q + i) * CL + lane];
    return;
  }
  // Inverse of this wave's 16 x 16 diagonal block [A 0; B C]: lane 8 t + c < 16 has
  // column c of the inverse of A (t = 0) or C (t = 1), then -C^-1 (B A^-1) by MFMA
  {
    const int t = lane / 8 % 2, o = 8 * t, cl = lane % 8, r0 = 16 * q + o;
    double* iv = Inv[q];
    double s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = cl == i ? 1.0 : 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      s[k] *= rdg[r0 + k];
#pragma unroll
      for (int i = k + 1; i < 8; ++i) s[i] -= s[k] * Ls[(r0 + k) * CL + r0 + i];
    }
    if (lane < 16)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        iv[(o + cl) * CI + o + i] = s[i];
        iv[(o + cl) * CI + 8 - o + i] = 0.0;
      }
    wave_lds_fence();
    v4d ba[1] = {v4d{0, 0, 0, 0}}, cba[1] = {v4d{0, 0, 0, 0}};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const double lb = m >= 8 ? Ls[(16 * q + 4 * k + g) * CL + 16 * q + m] : 0.0;
      ba[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(lb, iv[m * CI + 4 * k + g], ba[0], 0, 0, 0);
    }
#pragma unroll
    for (int k = 2; k < 4; ++k)
      cba[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(iv[(4 * k + g) * CI + m], ba[0][k], cba[0], 0, 0, 0);
    mfma_settle_f64<1>(cba);
    if (m < 8) {
      iv[m * CI + 8 + g] = -cba[0][2];
      iv[m * CI + 12 + g] = -cba[0][3];
    }
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    v4d lx = v4d{0, 0, 0, 0};
#pragma unroll
    for (int p = 0; p < b; ++p)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        lx = __builtin_amdgcn_mfma_f64_16x16x4f64(-Ls[(16 * p + 4 * s + g) * CL + 16 * b + m], x[p][s], lx, 0, 0, 0);
    x[b] += lx;
    double inv[4];
    v4d t = v4d{0, 0, 0, 0}, r = x[b];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      inv[s] = Inv[b][(4 * s + g) * CI + m];
      t = __builtin_amdgcn_mfma_f64_16x16x4f64(inv[s], x[b][s], t, 0, 0, 0);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
      r = __builtin_amdgcn_mfma_f64_16x16x4f64(-Ls[(16 * b + 4 * s + g) * CL + 16 * b + m], t[s], r, 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 4; ++s) t = __builtin_amdgcn_mfma_f64_16x16x4f64(inv[s], r[s], t, 0, 0, 0);
    x[b] = t;
  }
  mfma_settle_f64<4>(x);
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int xc = 16 * b + 4 * v + g, xr = 16 * q + m;
      if (xr < h && xc < w) Xp[xr + xc * xs] = x[b][v];
    }
}

// Workgroup 0: the panel's factored diagonal tile from its staging copy into
// A.  The next mt (mt + 1) / 2 workgroups: A_ij -= L_i L_j^T for the tiles
// (i, j), kp < j <= i, of the diagonal block (lower triangle only on diagonal
// tiles), the last mt (with a right-hand side) the same for y as one more row.
// One 64 x 64 tile per workgroup on transposed 16 x 16 MFMA tiles, wave q the
// rows 16 q ..; all loads in flight at once, the products in a rolled loop.
// 19 -> 8 us in a block of 1024 columns (4 x 4 register tiles before); 22 on average in
// one of 4096.
__global__ __launch_bounds__(256) void chol_update_kernel(double* A, int64_t lda, int64_t stride, int64_t d0,
                                                          int64_t kb, int kp, const double* __restrict__ dtile,
                                                          double* y) {
  __shared__ double Li[CT * CL], Lj[CT * CL];
  double* Ab = A + (int64_t)blockIdx.y * stride;
  const int tid = threadIdx.x, lane = tid % WAVE, g = lane / 16, m = lane % 16;
  const int q = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int64_t p0 = d0 + (int64_t)kp * CT;
  const int w = (int)(kb - (int64_t)kp * CT < CT ? kb - (int64_t)kp * CT : CT);
  if (blockIdx.x == 0) {  // the panel's factored diagonal tile into A (no tile below reads it)
    const double* dt = dtile + (int64_t)blockIdx.y * CT * CT;
    for (int e = tid; e < CT * CT; e += 256) {
      const int r = e % CT, c = e / CT;
      if (r < w && c < w && r >= c) Ab[(p0 + r) + (p0 + c) * lda] = dt[c * CT + r];
    }
    return;
  }
  const int mt = (int)((kb + CT - 1) / CT) - kp - 1, tiles = mt * (mt + 1) / 2;
  const bool yrow = (int)blockIdx.x > tiles;
  int ti, tj;
  if (yrow) {
    ti = mt;
    tj = (int)blockIdx.x - 1 - tiles;
  } else {
    tile_of(blockIdx.x - 1, ti, tj);
  }
  const int64_t ri = d0 + (int64_t)(kp + 1 + ti) * CT, rj = d0 + (int64_t)(kp + 1 + tj) * CT;
  const int hi = yrow ? 1 : (int)(kb - (ri - d0) < CT ? kb - (ri - d0) : CT);
  const int hj = (int)(kb - (rj - d0) < CT ? kb - (rj - d0) : CT);
  const double* Rp = yrow ? y + p0 : Ab + ri + p0 * lda;
  const double* Jp = Ab + rj + p0 * lda;
  double* Cp = yrow ? y + rj : Ab + ri + rj * lda;
  const int64_t cs = yrow ? 1 : lda;
  const int row = 16 * q + m;
  double lj[16], li[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int l = 4 * i + q;
    lj[i] = load_or_zero(Jp, lane + l * lda, lane < hj && l < w);
    li[i] = load_or_zero(Rp, lane + l * cs, lane < hi && l < w);
  }
  v4d c[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int col = 16 * b + 4 * v + g;
      c[b][v] = load_or_zero(Cp, row + col * cs, row < hi && col < hj && (ti != tj || row >= col));
    }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    Lj[(4 * i + q) * CL + lane] = -lj[i];
    Li[(4 * i + q) * CL + lane] = li[i];
  }
  __syncthreads();
  if (16 * q >= hi) return;
  // the products are summed by themselves and taken off at once: 64 roundings the
  // size of the sum instead of the size of A_ij
  v4d ll[4] = {v4d{0, 0, 0, 0}, v4d{0, 0, 0, 0}, v4d{0, 0, 0, 0}, v4d{0, 0, 0, 0}};
#pragma unroll 2
  for (int s = 0; s < 16; ++s) {
    const double l = Li[(4 * s + g) * CL + row];
#pragma unroll
    for (int b = 0; b < 4; ++b)
      ll[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(Lj[(4 * s + g) * CL + 16 * b + m], l, ll[b], 0, 0, 0);
  }
  mfma_settle_f64<4>(ll);
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int col = 16 * b + 4 * v + g;
      if (row < hi && col < hj && (ti != tj || row >= col)) Cp[row + col * cs] = c[b][v] + ll[b][v];
    }
}

// y -= L21 z for the m rows below a diagonal block (L21: m x kb, column-major):
// 64 rows per workgroup, the columns dealt to its 16 waves
__global__ __launch_bounds__(1024) void chol_fwd_gemv_kernel(const double* __restrict__ L21, int64_t lda, int64_t m,
                                                             int64_t kb, const double* __restrict__ z,
                                                             double* __restrict__ y) {
  __shared__ double sh[16][WAVE];
  const int lane = threadIdx.x % WAVE, q = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int64_t i = (int64_t)blockIdx.x * WAVE + lane;
  double a = 0.0;
  if (i < m)
#pragma unroll 8
    for (int64_t c = q; c < kb; c += 16) a += L21[i + c * lda] * z[c];
  sh[q][lane] = a;
  __syncthreads();
  if (q == 0 && i < m) {
    a = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) a += sh[k][lane];
    y[i] -= a;
  }
}

// One 64-row step of x = L^-T y from the last block up: x_b = L_bb^-T y_b, then
// y_j -= L_bj^T x_b for the blocks j < b, one per workgroup.  Every workgroup
// solves the 64 x 64 triangle (a chain of 64 lane reads; cheaper than a launch
// between); x goes to its own vector, since the others still read y_b.  The
// column sums halve their values with every step of the butterfly.
// 5.8 us a step; with y' = L^-1 y in the factorisation, n = 4096: 2.0 -> 0.4 ms
// against a library's substitutions, n = 272: 0.21 -> 0.03 ms.
__global__ __launch_bounds__(256) void chol_back_kernel(const double* __restrict__ A, int64_t n, int b,
                                                        double* y, double* __restrict__ x) {
  __shared__ double Ls[CT * (CT + 1)];
  __shared__ double xb[CT];
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int q = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int64_t p0 = (int64_t)b * CT, j0 = (int64_t)blockIdx.x * CT + 16 * q;
  const int w = (int)(n - p0 < CT ? n - p0 : CT);
  double p[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int c = 16 * q + i;
    p[i] = load_or_zero(A + p0 + p0 * n, lane + c * n, lane < w && lane >= c);
    if (lane == c && lane >= w) p[i] = 1.0;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) Ls[(16 * q + i) * (CT + 1) + lane] = p[i];
#pragma unroll
  for (int i = 0; i < 16; ++i) p[i] = load_or_zero(A + p0, lane + (j0 + i) * n, b > 0 && lane < w);
  __syncthreads();
  if (q == 0) {
    double z = lane < w ? y[p0 + lane] : 0.0, xi = 0.0;
    const double rd = 1.0 / Ls[lane * (CT + 1) + lane];
#pragma unroll 8
    for (int i = CT - 1; i >= 0; --i) {
      const double v = readlane_f64(z * rd, i);
      xi = lane == i ? v : xi;
      z -= Ls[lane * (CT + 1) + i] * v;  // zero above the diagonal; z of lane i is not used again
    }
    xb[lane] = xi;
    if (blockIdx.x == 0 && lane < w) x[p0 + lane] = xi;
  }
  if (b == 0) return;
  __syncthreads();
  const double xr = xb[lane];
#pragma unroll
  for (int i = 0; i < 16; ++i) p[i] *= xr;
  halve_columns<8, 4>(p, lane);
  halve_columns<4, 4>(p, lane);
  halve_columns<2, 4>(p, lane);
  halve_columns<1, 4>(p, lane);
  double s = p[0];
  s += __shfl_xor(s, 1, WAVE);
  s += __shfl_xor(s, 2, WAVE);
  if (lane % 4 == 0) y[j0 + lane / 4] -= s;
}

// y (batch 1): L^-1 y on return
static int blocked_potrf(rocblas_handle h, hipStream_t st, int64_t n, double* A, int64_t stride, int batch,
                         int32_t* info, int64_t info_stride, double* dtile, double* y = nullptr) {
  QTX_REQUIRE(y == nullptr || batch == 1, "one right-hand side per factorisation");
  const double one = 1.0, minus_one = -1.0;
  const rocblas_int ld = (rocblas_int)n;
  int b = 0;
  for (int64_t k = 0, kb; k < n; k += kb, ++b) {
    kb = chol_block(n - k, batch);
    const int nt = (int)((kb + CT - 1) / CT);
    for (int kp = 0; kp < nt; ++kp) {
      hipLaunchKernelGGL(chol_panel_kernel, dim3((unsigned)(nt - kp + (y ? 1 : 0)), (unsigned)batch), dim3(256), 0, st,
                         A, (int64_t)n, stride, k, kb, kp, info + b, info_stride, dtile, y);
      const int m = nt - kp - 1;
      hipLaunchKernelGGL(chol_update_kernel, dim3((unsigned)(1 + m * (m + 1) / 2 + (y ? m : 0)), (unsigned)batch),
                         dim3(256), 0, st, A, (int64_t)n, stride, k, kb, kp, (const double*)dtile, y);
    }
    QTX_LAUNCH_CHECK();
    const int64_t m = n - k - kb;
    if (m == 0) break;
    // one call per matrix: the strided-batched forms of these two routines
    // run on much slower non-GEMM kernels at these sizes
    for (int bi = 0; bi < batch; ++bi) {
      double* Akk = A + bi * stride + k * n + k;
      double* Apan = Akk + kb;
      int rc = rb(rocblas_dtrsm(h, rocblas_side_right, rocblas_fill_lower, rocblas_operation_transpose,
                                rocblas_diagonal_non_unit, (rocblas_int)m, (rocblas_int)kb, &one, Akk, ld, Apan, ld),
                  "rocblas_dtrsm");
      if (rc) return rc;
      double* A22 = A + bi * stride + (k + kb) * n + (k + kb);
      rc = rb(rocblas_dsyrk(h, rocblas_fill_lower, rocblas_operation_none, (rocblas_int)m, (rocblas_int)kb,
                            &minus_one, Apan, ld, &one, A22, ld),
              "rocblas_dsyrk");
      if (rc) return rc;
      if (y) {
        hipLaunchKernelGGL(chol_fwd_gemv_kernel, dim3(nblk(m, WAVE)), dim3(1024), 0, st, (const double*)Apan, n, m, kb,
                           (const double*)(y + k), y + k + kb);
        QTX_LAUNCH_CHECK();
      }
    }
  }
  return QTX_OK;
}

// x = L^-T y; y is overwritten
static int chol_back(hipStream_t st, int64_t n, const double* L, double* y, double* x) {
  for (int64_t b = (n + CT - 1) / CT - 1; b >= 0; --b)
    hipLaunchKernelGGL(chol_back_kernel, dim3((unsigned)std::max<int64_t>(1, b)), dim3(256), 0, st, L, n, (int)b, y, x);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

// ---------------------------------------------------------------- triangular inverse
// L^-1 in place of a lower-triangular L (column-major, leading dimension ld).
// The kTriLeaf-wide diagonal blocks are inverted by one batched rocSOLVER
// call; the blocks are then joined bottom-up: for L = [A 0; B C] with A and C
// already inverted, the lower-left block becomes -C^-1 (B A^-1).  Both
// triangular products run as DGEMMs over a leaf-aligned split of the triangle
// (a leaf diagonal block multiplies as a full block, zeroed above its
// diagonal first), so nearly all of the n^3 / 3 flops are large DGEMMs: 29 ms
// at n = 16384 on MI355X against 43 ms for rocsolver_dtrtri, with the same
// results to rounding (max difference 6e-16 relative).  W holds the products'
// intermediate B A^-1: at least (n - n/2) x n/2 doubles at leading dimension
// ld.
constexpr int64_t kTriLeaf = 1024;

__global__ __launch_bounds__(256) void zero_leaf_upper_kernel(double* A, int64_t n, int64_t ld) {
  const int64_t o = (int64_t)blockIdx.y * kTriLeaf;
  const int64_t m = (n - o < kTriLeaf) ? n - o : kTriLeaf;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < m * m; e += (int64_t)gridDim.x * 256) {
    const int64_t r = e % m, c = e / m;
    if (r < c) A[(o + r) + (o + c) * ld] = 0.0;
  }
}

// first failure of a chain of library calls; a device-memory size query
// answers with the size statuses, which count as success there
struct BlasChain {
  rocblas_handle h;
  rocblas_status st = rocblas_status_success;
  const char* what = nullptr;
  void operator()(rocblas_status s, const char* w) {
    const bool ok = s == rocblas_status_success || s == rocblas_status_size_increased ||
                    s == rocblas_status_size_unchanged;
    if (!ok && st == rocblas_status_success) {
      st = s;
      what = w;
    }
  }
};

// leaf-aligned split of m > kTriLeaf rows: the first part holds ceil(leaves / 2) leaves
static int64_t tri_split(int64_t m) {
  const int64_t nb = (m + kTriLeaf - 1) / kTriLeaf;
  return (nb + 1) / 2 * kTriLeaf;
}

static void tri_gemm(BlasChain& b, int64_t m, int64_t n, int64_t k, double alpha, const double* A, int64_t lda,
                     const double* B, int64_t ldb, double beta, double* C, int64_t ldc) {
  b(rocblas_dgemm(b.h, rocblas_operation_none, rocblas_operation_none, (rocblas_int)m, (rocblas_int)n,
                  (rocblas_int)k, &alpha, A, (rocblas_int)lda, B, (rocblas_int)ldb, &beta, C, (rocblas_int)ldc),
    "rocblas_dgemm");
}

// W = alpha X T, X: r x t, T: t x t lower triangular starting at a leaf boundary
static void tri_mul_right(BlasChain& b, int64_t r, int64_t t, double alpha, const double* X, int64_t ldx,
                          const double* T, int64_t ldt, double* W, int64_t ldw) {
  if (t <= kTriLeaf) {
    tri_gemm(b, r, t, t, alpha, X, ldx, T, ldt, 0.0, W, ldw);
    return;
  }
  const int64_t t1 = tri_split(t), t2 = t - t1;  // T = [P 0; Q R], X = [X1 X2]
  tri_mul_right(b, r, t1, alpha, X, ldx, T, ldt, W, ldw);                         // X1 P
  tri_gemm(b, r, t1, t2, alpha, X + t1 * ldx, ldx, T + t1, ldt, 1.0, W, ldw);     // + X2 Q
  tri_mul_right(b, r, t2, alpha, X + t1 * ldx, ldx, T + t1 + t1 * ldt, ldt, W + t1 * ldw, ldw);  // X2 R
}

// W = alpha T X, T: t x t lower triangular starting at a leaf boundary, X: t x c
static void tri_mul_left(BlasChain& b, int64_t t, int64_t c, double alpha, const double* T, int64_t ldt,
                         const double* X, int64_t ldx, double* W, int64_t ldw) {
  if (t <= kTriLeaf) {
    tri_gemm(b, t, c, t, alpha, T, ldt, X, ldx, 0.0, W, ldw);
    return;
  }
  const int64_t t1 = tri_split(t), t2 = t - t1;  // T = [P 0; Q R], X = [X1; X2]
  tri_mul_left(b, t1, c, alpha, T, ldt, X, ldx, W, ldw);                                  // P X1
  tri_mul_left(b, t2, c, alpha, T + t1 + t1 * ldt, ldt, X + t1, ldx, W + t1, ldw);        // R X2
  tri_gemm(b, t2, c, t1, alpha, T + t1, ldt, X, ldx, 1.0, W + t1, ldw);                   // + Q X1
}

static void tri_join(BlasChain& b, double* A, int64_t ld, int64_t m, double* W) {
  if (m <= kTriLeaf) return;
  const int64_t m1 = tri_split(m), m2 = m - m1;
  tri_join(b, A, ld, m1, W);
  tri_join(b, A + m1 + m1 * ld, ld, m2, W);
  tri_mul_right(b, m2, m1, 1.0, A + m1, ld, A, ld, W, ld);                    // W = B A^-1
  tri_mul_left(b, m2, m1, -1.0, A + m1 + m1 * ld, ld, W, ld, A + m1, ld);     // B = -C^-1 W
}

// info[i] (i < number of leaves) receives rocSOLVER's status of leaf i.  With
// query set, only the library calls are made (inside a device-memory size
// query): no kernel runs
static int tri_inverse(rocblas_handle h, hipStream_t st, int64_t n, double* A, int64_t ld, double* W,
                       int32_t* info, bool query) {
  BlasChain b{h};
  const int64_t full = n / kTriLeaf, rem = n % kTriLeaf;
  if (full)
    b(rocsolver_dtrtri_strided_batched(h, rocblas_fill_lower, rocblas_diagonal_non_unit, (rocblas_int)kTriLeaf, A,
                                       (rocblas_int)ld, (rocblas_stride)(kTriLeaf * ld + kTriLeaf), info,
                                       (rocblas_int)full),
      "rocsolver_dtrtri_strided_batched");
  if (rem)
    b(rocsolver_dtrtri(h, rocblas_fill_lower, rocblas_diagonal_non_unit, (rocblas_int)rem,
                       A + full * kTriLeaf * (ld + 1), (rocblas_int)ld, info + full),
      "rocsolver_dtrtri");
  if (full && !query) {
    hipLaunchKernelGGL(zero_leaf_upper_kernel, dim3(64, (unsigned)(full + (rem ? 1 : 0))), dim3(256), 0, st, A, n,
                       ld);
    QTX_LAUNCH_CHECK();
  }
  tri_join(b, A, ld, n, W);
  if (b.st != rocblas_status_success) return rb(b.st, b.what);
  return QTX_OK;
}

// tri_pass_kernel for this n (tri_pass_ok); part needs TP_GRID n doubles
template <bool SYM>
static int launch_tri_pass(hipStream_t st, const double* S, int64_t n, const double* X, double* part, double* dots) {
#define QTX_TP(RB, NC)                                                                                             \
  do {                                                                                                             \
    QTX_HIP(hipFuncSetAttribute((const void*)tri_pass_kernel<RB, NC, SYM>,                                         \
                                hipFuncAttributeMaxDynamicSharedMemorySize, tp_lds<NC>()));                    \
    hipLaunchKernelGGL((tri_pass_kernel<RB, NC, SYM>), dim3(TP_GRID), dim3(TP_THREADS), (tp_lds<NC>()), st, S, \
                       n, X, part, dots);                                                                          \
  } while (0)
  if (n <= 4096) QTX_TP(4, 4);
  else if (n <= 8192) QTX_TP(2, 8);
  else QTX_TP(1, 16);
#undef QTX_TP
  return QTX_OK;
}
static bool tri_pass_ok(int64_t n, bool sym) {
  return n >= (sym ? kTriPassSymMin : kTriPassMin) && n <= kTriPassMax;
}

// ---------------------------------------------------------------- phased solve
// A solve runs as three phases so that many solves on different streams can
// be driven from one host thread with batched host syncs
// (qtx_minsr_solve_many): every task's phase p is enqueued before any task's
// phase p + 1 reads results back.
//   phase 1: Gram (and for SR the right-hand side Obar^T ebar); CHOL_SHIFT:
//            shift, factorisation and both substitutions; EIGH_PINV: the first
//            Lanczos steps.
//   phase 2: EIGH_PINV: read the Lanczos coefficients (sync), extend until the
//            largest Ritz value settles, then syrk + three (potrf, refinement)
//            for the partial fractions; dsyevd where that route does not apply.
//   phase 3: read the factorisation status (sync); dsyevd fallback; the update
//            vector x = Obar^T y.
// All phases of different tasks overlap on their streams (the factorisations
// too, unless QTX_SERIAL_FACTOR=1).  A panel kernel of the blocked Cholesky
// once stored its factored diagonal tile into the matrix while other
// workgroups of the same launch could still be reading the unfactored tile;
// delayed workgroups — common when other tasks occupy the GPU — then factored
// garbage (non-positive pivots in 249 of 640 overlapped solves); the tile is
// now staged and stored by the next launch.
// Chebyshev coefficients of h(mu) = g(sigma mu / (1 - mu)), g(v) = v^5 /
// (v^6 + c^6), on [mu_lo, mu_max] (mu = mu_lo + (mu_max - mu_lo) (u + 1) / 2,
// u in [-1, 1]) from kChebNodes Chebyshev points (a discrete cosine
// transform); returns the number of terms kept, 0 when the series does not
// settle within kChebMax.
static int cheb_coeffs_raw(double c, double sigma, double mu_lo, double mu_max, std::vector<double>& a) {
  const int N = kChebNodes;
  std::vector<double> f(N);
  const double pi = 3.14159265358979323846;
  for (int j = 0; j < N; ++j) {
    const double u = cos(pi * (j + 0.5) / N), mu = mu_lo + (mu_max - mu_lo) * (u + 1.0) * 0.5;
    const double tt = sigma * mu / ((1.0 - mu) * c);  // v / c, negative below mu = 0
    const double t5 = tt * tt * tt * tt * tt;
    f[j] = t5 / (t5 * tt + 1.0) / c;
  }
  const int K = kChebMax + 8;
  a.assign(K, 0.0);
  for (int j = 0; j < N; ++j) {  // cos(k theta_j) by the three-term recurrence
    const double c1 = cos(pi * (j + 0.5) / N);
    double ckm = 1.0, ck = c1;
    a[0] += f[j];
    a[1] += f[j] * c1;
    for (int k = 2; k < K; ++k) {
      const double cn = 2.0 * c1 * ck - ckm;
      a[k] += f[j] * cn;
      ckm = ck;
      ck = cn;
    }
  }
  double amax = 0.0;
  for (int k = 0; k < K; ++k) {
    a[k] *= (k == 0 ? 1.0 : 2.0) / N;
    amax = std::max(amax, fabs(a[k]));
  }
  for (int k = 8; k < kChebMax; ++k) {
    bool small = true;
    for (int m = k; m < k + 8; ++m) small = small && fabs(a[m]) < kChebTol * amax;
    if (small) {
      a.resize(k);
      return k;
    }
  }
  return 0;
}

// sigma = c: the series of c h depends on mu_max = 1 / (1 + rel) alone (rel =
// c / lambda_max), so it is computed once per rel and thread
static int cheb_coeffs(double c, double rel, std::vector<double>& a) {
  static thread_local std::vector<std::pair<double, std::vector<double>>> cache;
  for (const auto& e : cache)
    if (e.first == rel) {
      a = e.second;
      for (double& v : a) v /= c;
      return (int)a.size();
    }
  std::vector<double> u;
  const int k = cheb_coeffs_raw(1.0, 1.0, -kChebMargin, 1.0 / (1.0 + rel), u);
  if (k == 0) return 0;
  if (cache.size() >= 16) cache.erase(cache.begin());
  cache.emplace_back(rel, u);
  a = u;
  for (double& v : a) v /= c;
  return k;
}

struct Task {
  qtx_minsr_task* io = nullptr;
  hipStream_t st = nullptr;
  SolveWs w{};
  char* blas_ws = nullptr;  // QTX_SOLVE_BLAS_WS: rocBLAS scratch = the workspace past the library's own part
  size_t blas_bytes = 0;
  bool minnorm = false;
  int64_t n = 0;
  bool failed = false;
  bool need_syevd = false;  // phase 2 runs the dsyevd route
  bool pf = false;          // partial-fraction factorisations enqueued
  bool cf = false;          // shifted Cholesky route enqueued (small cutoffs)
  bool cheb = false;        // Chebyshev route enqueued
  int cheb_terms = 0;
  double c = 0.0, rel = 0.0;  // the cutoff and c / lambda_max
  int mcap = 0, done = 0;   // Lanczos steps available / enqueued
  double lmax = 0.0;
  int lanczos = 0;
  int path = -1, fallback = 0;
};

// whether the weights' values choose the route: only below a cutoff of 1e-5 (a copy of
// the flag costs about 20 us)
static bool ones_asked(const Task& t) { return t.minnorm && t.io->r && !(t.io->rtol >= 1e-5); }

static int task_fail(Task& t, int rc) {
  t.failed = true;
  t.io->status = rc;
  return rc;
}

static int lanczos_enqueue(Task& t, rocblas_handle h, int to) {
  (void)h;
  double* alpha = t.w.ab;
  double* beta = t.w.ab + kLanczosMax;
  const unsigned gm = (unsigned)((t.n + 3) / 4);
  for (int j = t.done; j < to; ++j) {
    double* v = t.w.V + (j % 3) * t.n;
    double* vp = t.w.V + ((j + 2) % 3) * t.n;
    double* vn = t.w.V + ((j + 1) % 3) * t.n;
    if (tri_pass_ok(t.n, true)) {  // T2 is free until the factorisation
      int rc = launch_tri_pass<true>(t.st, t.w.T, t.n, v, t.w.T2, t.w.R);
      if (rc) return rc;
      hipLaunchKernelGGL(tp_sum_kernel, dim3(nblk(t.n, TP_COLS)), dim3(1024), 0, t.st, t.w.T2, t.w.R, t.n, t.w.w);
    } else {
      hipLaunchKernelGGL(matvec_rows_kernel<1>, dim3(gm), dim3(256), 0, t.st, t.w.T, t.n, v, t.w.w);
    }
    const auto step = t.n <= 1024    ? lanczos_step_kernel<1>
                      : t.n <= 4096  ? lanczos_step_kernel<4>
                      : t.n <= 16384 ? lanczos_step_kernel<16>
                                     : lanczos_step_kernel<0>;
    hipLaunchKernelGGL(step, dim3(1), dim3(1024), 0, t.st, t.n, j, t.w.w, v, vp, vn, alpha, beta);
  }
  QTX_LAUNCH_CHECK();
  t.done = to;
  return QTX_OK;
}

template <typename TI>
static int phase1(Task& t, rocblas_handle h) {
  qtx_minsr_task& io = *t.io;
  const TI* O = (const TI*)io.O;
  int rc;
  if (t.minnorm) {
    rc = launch_gram_nt<TI>(t.st, io.gram, O, io.mean, io.r, io.ns, io.np, t.w.T, t.w.split);
    if (rc) return rc;
    hipLaunchKernelGGL(copy_f64_kernel, dim3(nblk(io.ns, 256)), dim3(256), 0, t.st, io.ebar, t.w.y, io.ns);
  } else {
    // S = Obar^T Obar; beyond kGramTnMax Obar formed in FP64 a row block at a time,
    // each block accumulated by one rocBLAS DGEMM (a row-major rows x np block is
    // the column-major np x rows matrix B, S += B B^T)
    if (io.np <= kGramTnMax) {
      if ((rc = launch_gram_tn<TI>(t.st, O, io.mean, io.r, io.ns, io.np, t.w.T))) return rc;
    } else {
      const int64_t rows = obar_rows(io.ns, io.np);
      const double one = 1.0, zero = 0.0;
      for (int64_t s0 = 0; s0 < io.ns; s0 += rows) {
        const int64_t nr = std::min(rows, io.ns - s0), tot = nr * io.np;
        hipLaunchKernelGGL(form_obar_kernel<TI>, dim3((unsigned)std::min<int64_t>((tot + 255) / 256, kGridCap)),
                           dim3(256), 0, t.st, O + s0 * io.np, io.mean, io.r ? io.r + s0 : nullptr, nr, io.np,
                           1.0 / (double)io.ns, t.w.obar);
        QTX_LAUNCH_CHECK();
        rc = rb(rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_transpose, (rocblas_int)io.np,
                              (rocblas_int)io.np, (rocblas_int)nr, &one, t.w.obar, (rocblas_int)io.np, t.w.obar,
                              (rocblas_int)io.np, s0 ? &one : &zero, t.w.T, (rocblas_int)io.np),
                "rocblas_dgemm");
        if (rc) return rc;
      }
    }
    rc = launch_obar_t_y<TI>(t.st, O, io.mean, io.r, io.ebar, io.ns, io.np, t.w.y);  // F = Obar^T ebar
    if (rc) return rc;
  }
  const rocblas_int ni = (rocblas_int)t.n;
  const int mode = base_mode(io.mode);
  if (mode == QTX_SOLVE_CHOL_SHIFT) {
    hipLaunchKernelGGL(shift_diag_kernel, dim3(1), dim3(1024), 0, t.st, t.w.T, t.n, io.rshift, io.ashift,
                       t.w.scalars);
    QTX_LAUNCH_CHECK();
    hipLaunchKernelGGL(fill_i32_kernel, dim3(nblk(3 * kInfoPerFactor, 256)), dim3(256), 0, t.st, t.w.info,
                       (int64_t)(3 * kInfoPerFactor), 0);
    rc = blocked_potrf(h, t.st, t.n, t.w.T, 0, 1, t.w.info, kInfoPerFactor, t.w.dtile, t.w.y);
    if (rc) return rc;
    std::swap(t.w.y, t.w.z);
    return chol_back(t.st, t.n, t.w.T, t.w.z, t.w.y);
  }
  if (mode == QTX_SOLVE_EIGH_PINV_DIRECT) {
    t.need_syevd = true;
    return QTX_OK;
  }
  if (io.tol_snr > kSnrMin) {  // the truncation needs the eigenvectors
    t.fallback = 5;
    t.need_syevd = true;
    return QTX_OK;
  }
  // lambda_max = max |eigenvalue| of the PSD T by Lanczos (three-term
  // recurrence; the largest Ritz value is checked every 32 steps)
  hipLaunchKernelGGL(lanczos_init_kernel, dim3(1), dim3(1024), 0, t.st, t.n, t.w.V, t.w.ab + kLanczosMax);
  t.mcap = (int)(t.n < kLanczosMax ? t.n : kLanczosMax);
  // whether the weights are all one, for the small-cutoff route of phase 2
  if (ones_asked(t))
    hipLaunchKernelGGL(all_ones_kernel, dim3(1), dim3(1024), 0, t.st, io.r, io.ns, t.w.scalars + 2);
  // convergence checks every 16 steps when one product streams more than
  // 512 MB of T (n > 8192: 16 products cost far more than the host round
  // trip of a check; a VMC Gram's top eigenvalue, well separated, settles
  // within 8 steps), else after 48 and then every 32
  const int first = t.n > 8192 ? 16 : 48;
  return lanczos_enqueue(t, h, t.mcap < first ? t.mcap : first);
}

static int snr_syevd(Task& t, rocblas_handle h) {
  qtx_minsr_task& io = *t.io;
  SnrRows rows{io.o_dtype, io.O, io.mean, io.r, io.ebar, io.ns, io.np};
  return pinv_syevd(t.st, h, t.n, io.rtol, io.atol, t.w, io.tol_snr, t.minnorm ? nullptr : &rows);
}

// Partial-fraction route: T^2 by dsyrk, the three quadratics (T - a_k)^2 + b_k^2
// factored together, and iterative refinement of the complex shifted systems
// against T itself.
static int pf_enqueue(Task& t, rocblas_handle h, double c, double rel) {
  // refinement contracts by about 4 u / rel^2 per pass (4.4e-8 at rel = 1e-4,
  // 4.4e-6 at 1e-5): two passes reach ~1e-15 for rel >= 1e-4, three for 1e-5
  const int iters = rel >= 1e-4 ? 2 : (rel >= 1e-5 ? 3 : 4);
  const rocblas_int ni = (rocblas_int)t.n;
  const double one = 1.0, zero = 0.0;
  const unsigned gb = (unsigned)nblk(t.n, 256);
  const unsigned gm = (unsigned)((t.n + 3) / 4);
  int rc = rb(rocblas_dsyrk(h, rocblas_fill_lower, rocblas_operation_none, ni, ni, &one, t.w.T, ni, &zero,
                            t.w.T2, ni),
              "rocblas_dsyrk");
  if (rc) return rc;
  hipLaunchKernelGGL(fill_i32_kernel, dim3(nblk(3 * kInfoPerFactor, 256)), dim3(256), 0, t.st, t.w.info,
                     (int64_t)(3 * kInfoPerFactor), 0);
  // pole k = c e^{i pi (2k+1)/6}: quadratic k into matrix k of the T2 block,
  // k = 0 last because it overwrites T^2 in place
  const int64_t nn = t.n * t.n;
  double pa[3], pb[3];
  for (int k = 0; k < 3; ++k) {
    const double th = 3.14159265358979323846 * (2 * k + 1) / 6.0;
    pa[k] = (k == 1) ? 0.0 : c * cos(th);
    pb[k] = c * sin(th);
  }
  const unsigned gq = (unsigned)std::min<int64_t>((nn + 255) / 256, kGridCap);
  for (int k : {1, 2, 0}) {
    hipLaunchKernelGGL(form_quad_kernel, dim3(gq), dim3(256), 0, t.st, t.w.T2, t.w.T, t.n, 2.0 * pa[k], c * c,
                       t.w.T2 + k * nn);
    QTX_LAUNCH_CHECK();
  }
  rc = blocked_potrf(h, t.st, t.n, t.w.T2, nn, 3, t.w.info, kInfoPerFactor, t.w.dtile);
  if (rc) return rc;
  // iterative refinement of the three complex systems (T - p_k) z = y,
  // the inner solves batched over the three factors, the products with T
  // over all six vectors in one pass
  for (int k = 0; k < 3; ++k)
    hipLaunchKernelGGL(refine_init_kernel, dim3(gb), dim3(256), 0, t.st, t.w.y, t.n, t.w.R + 2 * k * t.n,
                       t.w.Z + 2 * k * t.n);
  for (int it = 0; it < iters; ++it) {
    rc = rb(rocblas_dtrsm_strided_batched(h, rocblas_side_left, rocblas_fill_lower, rocblas_operation_none,
                                          rocblas_diagonal_non_unit, ni, 2, &one, t.w.T2, ni, nn, t.w.R, ni,
                                          2 * t.n, 3),
            "rocblas_dtrsm_strided_batched");
    if (rc) return rc;
    rc = rb(rocblas_dtrsm_strided_batched(h, rocblas_side_left, rocblas_fill_lower, rocblas_operation_transpose,
                                          rocblas_diagonal_non_unit, ni, 2, &one, t.w.T2, ni, nn, t.w.R, ni,
                                          2 * t.n, 3),
            "rocblas_dtrsm_strided_batched");
    if (rc) return rc;
    hipLaunchKernelGGL(matvec_rows_kernel<6>, dim3(gm), dim3(256), 0, t.st, t.w.T, t.n, t.w.R, t.w.TW);
    for (int k = 0; k < 3; ++k)
      hipLaunchKernelGGL(refine_update_kernel, dim3(gb), dim3(256), 0, t.st, t.w.R + 2 * k * t.n,
                         t.w.TW + 2 * k * t.n, t.n, pa[k], pb[k], t.w.Z + 2 * k * t.n);
    if (it + 1 < iters) {
      hipLaunchKernelGGL(matvec_rows_kernel<6>, dim3(gm), dim3(256), 0, t.st, t.w.T, t.n, t.w.Z, t.w.TW);
      for (int k = 0; k < 3; ++k)
        hipLaunchKernelGGL(refine_residual_kernel, dim3(gb), dim3(256), 0, t.st, t.w.y, t.w.Z + 2 * k * t.n,
                           t.w.TW + 2 * k * t.n, t.n, pa[k], pb[k], t.w.R + 2 * k * t.n);
    }
  }
  for (int k = 0; k < 3; ++k)
    hipLaunchKernelGGL(refine_accum_kernel, dim3(gb), dim3(256), 0, t.st, t.w.Z + 2 * k * t.n, t.n, k == 0 ? 1 : 0,
                       t.w.x);
  QTX_LAUNCH_CHECK();
  t.pf = true;
  return QTX_OK;
}

static int phase2(Task& t, rocblas_handle h) {
  qtx_minsr_task& io = *t.io;
  if (base_mode(io.mode) == QTX_SOLVE_CHOL_SHIFT) return QTX_OK;
  if (!t.need_syevd) {
    std::vector<double> ha(kLanczosMax), hb(kLanczosMax + 1);
    double lmax = 0.0;
    int msteps = 0;
    bool bad = false;
    double ones = io.r ? 0.0 : 1.0;  // read with the coefficients: no further wait
    if (ones_asked(t))
      QTX_HIP(hipMemcpyAsync(&ones, t.w.scalars + 2, sizeof(double), hipMemcpyDeviceToHost, t.st));
    for (;;) {
      QTX_HIP(hipMemcpyAsync(ha.data(), t.w.ab, (size_t)t.done * 8, hipMemcpyDeviceToHost, t.st));
      QTX_HIP(hipMemcpyAsync(hb.data(), t.w.ab + kLanczosMax, (size_t)(t.done + 1) * 8, hipMemcpyDeviceToHost, t.st));
      QTX_HIP(hipStreamSynchronize(t.st));
      int m = t.done;
      bool exact = false;
      for (int j = 0; j < t.done; ++j) {
        if (!std::isfinite(ha[j]) || !std::isfinite(hb[j + 1])) {
          bad = true;
          break;
        }
        if (hb[j + 1] == 0.0) {  // invariant Krylov subspace: the Ritz values are exact
          m = j + 1;
          exact = true;
          break;
        }
      }
      if (bad) break;
      lmax = tridiag_max_eig(ha.data(), hb.data(), m);
      msteps = m;
      if (exact || t.done >= t.mcap) break;
      double prev = tridiag_max_eig(ha.data(), hb.data(), m - 8);
      if (fabs(lmax - prev) <= 1e-14 * fabs(lmax)) break;
      const int more = t.n > 8192 ? 16 : 32;
      int rc = lanczos_enqueue(t, h, t.done + more < t.mcap ? t.done + more : t.mcap);
      if (rc) return rc;
    }
    t.lanczos = msteps;
    t.lmax = lmax;
    const double c = io.rtol * lmax + io.atol, rel = io.rtol + io.atol / lmax;  // c / lmax, exact for atol = 0
    if (bad) {
      t.fallback = 2;
    } else if (!(lmax > 0.0) || !std::isfinite(lmax)) {
      t.fallback = 3;
    } else if (!std::isfinite(c) || (!(rel >= 1e-5) && t.minnorm && ones == 0.0)) {
      t.fallback = 1;  // (reweighted MinSR: the null direction of T is not 1)
    }
    if (t.fallback) {
      t.need_syevd = true;
    } else if (!(rel >= 1e-5)) {
      // small cutoff: T_d x = b' by the shifted factorisation and refinement
      const rocblas_int ni = (rocblas_int)t.n;
      const double one = 1.0;
      const double mu_n = t.minnorm ? lmax / (double)t.n : 0.0;
      const int64_t nn = t.n * t.n;
      const unsigned gq = (unsigned)std::min<int64_t>((nn + 255) / 256, kGridCap);
      const unsigned gm = (unsigned)((t.n + 3) / 4);
      hipLaunchKernelGGL(fill_i32_kernel, dim3(nblk(3 * kInfoPerFactor, 256)), dim3(256), 0, t.st, t.w.info,
                         (int64_t)(3 * kInfoPerFactor), 0);
      hipLaunchKernelGGL(form_shifted_kernel, dim3(gq), dim3(256), 0, t.st, t.w.T, t.n, mu_n, kShiftCut * c, t.w.T2);
      QTX_LAUNCH_CHECK();
      int rc = blocked_potrf(h, t.st, t.n, t.w.T2, nn, 1, t.w.info, kInfoPerFactor, t.w.dtile);
      if (rc) return rc;
      double* r = t.w.R;
      double* z = t.w.R + t.n;
      double* p = t.w.R + 2 * t.n;
      double* q = t.w.TW;
      double* s = t.w.scalars + 4;
      hipLaunchKernelGGL(shifted_init_kernel, dim3(1), dim3(1024), 0, t.st, t.w.y, t.n, t.minnorm ? 1 : 0, t.w.z,
                         t.w.x, r, z);
      QTX_LAUNCH_CHECK();
      // L^-1 in place of L: each preconditioner application is then two
      // bandwidth-bound triangular products instead of two triangular solves
      // (a single-vector dtrsm at n = 16384 ran at ~10 ms)
      if ((rc = tri_inverse(h, t.st, t.n, t.w.T2, t.n, t.w.T2 + nn, t.w.info + kInfoPerFactor, false))) return rc;
      auto precondition = [&]() -> int {  // z <- G^-1 z = L^-T L^-1 z
        int rc2 = rb(rocblas_dtrmv(h, rocblas_fill_lower, rocblas_operation_none, rocblas_diagonal_non_unit, ni,
                                   t.w.T2, ni, z, 1),
                     "rocblas_dtrmv");
        if (rc2) return rc2;
        return rb(rocblas_dtrmv(h, rocblas_fill_lower, rocblas_operation_transpose, rocblas_diagonal_non_unit, ni,
                                t.w.T2, ni, z, 1),
                  "rocblas_dtrmv");
      };
      if ((rc = precondition())) return rc;
      hipLaunchKernelGGL(pcg_step2_kernel, dim3(1), dim3(1024), 0, t.st, r, z, t.n, 1, p, s);
      for (int it = 0; it < kShiftIters; ++it) {
        hipLaunchKernelGGL(matvec_rows_kernel<1>, dim3(gm), dim3(256), 0, t.st, t.w.T, t.n, p, q);
        hipLaunchKernelGGL(pcg_step1_kernel, dim3(1), dim3(1024), 0, t.st, q, p, t.n, mu_n, t.w.x, r, z, s);
        QTX_LAUNCH_CHECK();
        if ((rc = precondition())) return rc;
        hipLaunchKernelGGL(pcg_step2_kernel, dim3(1), dim3(1024), 0, t.st, r, z, t.n, 0, p, s);
      }
      hipLaunchKernelGGL(matvec_rows_kernel<1>, dim3(gm), dim3(256), 0, t.st, t.w.T, t.n, t.w.x, q);
      hipLaunchKernelGGL(pcg_check_kernel, dim3(1), dim3(1024), 0, t.st, t.w.z, q, t.w.x, t.n, mu_n,
                         t.w.scalars + 6);
      QTX_LAUNCH_CHECK();
      t.cf = true;
    }
    t.c = c;
    t.rel = rel;
    std::vector<double> ca;
    // sigma = c; mu_max from rel slightly reduced: the Ritz value may sit
    // just below lambda_max
    const double sigma = c;
    const double rel_s = rel / (1.0 + 1e-9);
    const double mu_max = 1.0 / (1.0 + rel_s), mu_lo = -kChebMargin;
    if (!t.need_syevd && !t.cf && (t.n >= kChebMinN || (io.mode & QTX_SOLVE_CHEB)) &&
        (t.cheb_terms = cheb_coeffs(c, rel_s, ca)) > 0) {
      // Chebyshev route: G = T + sigma I = L L^T, P = L^-1, then
      // x = sum_k a_k T_k(A) y with A = (2 / mu_max) (I - sigma P^T P) - I
      const int64_t nn = t.n * t.n;
      const unsigned gq = (unsigned)std::min<int64_t>((nn + 255) / 256, kGridCap);
      const unsigned gm = (unsigned)((t.n + 3) / 4);
      hipLaunchKernelGGL(fill_i32_kernel, dim3(nblk(3 * kInfoPerFactor, 256)), dim3(256), 0, t.st, t.w.info,
                         (int64_t)(3 * kInfoPerFactor), 0);
      hipLaunchKernelGGL(form_shifted_kernel, dim3(gq), dim3(256), 0, t.st, t.w.T, t.n, 0.0, -sigma, t.w.T2);
      QTX_LAUNCH_CHECK();
      int rc = blocked_potrf(h, t.st, t.n, t.w.T2, nn, 1, t.w.info, kInfoPerFactor, t.w.dtile);
      if (rc) return rc;
      if ((rc = tri_inverse(h, t.st, t.n, t.w.T2, t.n, t.w.T2 + nn, t.w.info + kInfoPerFactor, false))) return rc;
      const int nt = (int)((t.n + 63) / 64);
      hipLaunchKernelGGL(tri_mirror_kernel, dim3((unsigned)((int64_t)nt * (nt + 1) / 2)), dim3(256), 0, t.st, t.w.T2,
                         t.n, nt);
      double* B[2] = {t.w.R, t.w.R + t.n};  // t_k, t_{k +- 1}
      double* u = t.w.R + 2 * t.n;
      hipLaunchKernelGGL(copy_f64_kernel, dim3(nblk(t.n, 256)), dim3(256), 0, t.st, t.w.y, B[0], t.n);
      const double span = mu_max - mu_lo;
      const double alpha = (2.0 - mu_max - mu_lo) / span, beta = 2.0 * sigma / span;
      for (int k = 0; k + 1 < t.cheb_terms; ++k) {
        const double* tcur = B[k & 1];
        double* tprev = B[(k + 1) & 1];
        if (tri_pass_ok(t.n, false)) {  // the third of the n x n buffers is free here
          if ((rc = launch_tri_pass<false>(t.st, t.w.T2, t.n, tcur, t.w.T2 + 2 * nn, nullptr))) return rc;
          hipLaunchKernelGGL(tp_cheb_kernel, dim3(nblk(t.n, TP_COLS)), dim3(1024), 0, t.st, t.w.T2 + 2 * nn, t.n, tcur,
                             tprev, alpha, beta, ca[0], ca[k + 1], k == 0 ? 1 : 0, t.w.x);
          continue;
        }
        hipLaunchKernelGGL(tri_rows_kernel<true>, dim3(gm), dim3(256), 0, t.st, t.w.T2, t.n, tcur, u);
        hipLaunchKernelGGL(cheb_rows_kernel, dim3(gm), dim3(256), 0, t.st, t.w.T2, t.n, u, tcur, tprev, alpha, beta,
                           ca[0], ca[k + 1], k == 0 ? 1 : 0, t.w.x);
      }
      // |t_last|^2 and |y|^2 for the growth check
      hipLaunchKernelGGL(sq_norms_kernel, dim3(1), dim3(1024), 0, t.st, B[(t.cheb_terms - 1) & 1], t.w.y, t.n,
                         t.w.scalars + 4);
      QTX_LAUNCH_CHECK();
      t.cheb = true;
    } else if (!t.need_syevd && !t.cf) {
      int rc = pf_enqueue(t, h, c, rel);
      if (rc) return rc;
    }
  }
  if (t.need_syevd) {
    int rc = snr_syevd(t, h);
    if (rc < 0) return rc;
    t.path = 2;
  }
  return QTX_OK;
}

template <typename TI>
static int phase3(Task& t, rocblas_handle h) {
  qtx_minsr_task& io = *t.io;
  const bool chol = base_mode(io.mode) == QTX_SOLVE_CHOL_SHIFT;
  if (t.cheb) {
    std::vector<int32_t> info_h(2 * kInfoPerFactor);  // the factorisation's blocks, then the inverse's leaves
    double nrm[2];                                     // |t_last|^2, |y|^2
    QTX_HIP(hipMemcpyAsync(info_h.data(), t.w.info, info_h.size() * sizeof(int32_t), hipMemcpyDeviceToHost, t.st));
    QTX_HIP(hipMemcpyAsync(nrm, t.w.scalars + 4, sizeof(nrm), hipMemcpyDeviceToHost, t.st));
    QTX_HIP(hipStreamSynchronize(t.st));
    bool ok = true;
    for (int32_t v : info_h) ok = ok && (v == 0);
    const bool bounded = std::isfinite(nrm[0]) && nrm[0] <= kChebGrowth * kChebGrowth * nrm[1];
    if (ok && bounded) {
      hipLaunchKernelGGL(copy_f64_kernel, dim3(nblk(t.n, 256)), dim3(256), 0, t.st, t.w.x, t.w.y, t.n);
      QTX_LAUNCH_CHECK();
      t.path = 4;
    } else if (ok) {  // T has eigenvalues below the series' interval: partial fractions
      t.fallback = 8;
      int rc = pf_enqueue(t, h, t.c, t.rel);
      if (rc) return rc;
    } else {  // T and y are intact: take the dsyevd route
      t.fallback = 4;
      int rc = snr_syevd(t, h);
      if (rc < 0) return rc;
      t.path = 2;
    }
  }
  if (chol || t.pf) {
    std::vector<int32_t> info_h(3 * kInfoPerFactor);
    QTX_HIP(hipMemcpyAsync(info_h.data(), t.w.info, info_h.size() * sizeof(int32_t), hipMemcpyDeviceToHost, t.st));
    QTX_HIP(hipStreamSynchronize(t.st));
    int bad = -1;  // first diagonal block whose factorisation failed
    const int nslots = chol ? kInfoPerFactor : 3 * kInfoPerFactor;
    for (int i = 0; i < nslots && bad < 0; ++i)
      if (info_h[i] != 0) bad = i;
    if (chol) {
      if (bad >= 0)
        return fail(QTX_ESOLVER, "potrf failed in diagonal block " + std::to_string(bad) +
                                     " (info " + std::to_string(info_h[bad]) + ")");
      t.path = 0;
    } else if (bad >= 0) {  // T and y are intact: take the dsyevd route
      t.fallback = 4;
      int rc = snr_syevd(t, h);
      if (rc < 0) return rc;
      t.path = 2;
    } else {
      hipLaunchKernelGGL(copy_f64_kernel, dim3(nblk(t.n, 256)), dim3(256), 0, t.st, t.w.x, t.w.y, t.n);
      QTX_LAUNCH_CHECK();
      t.path = 1;
    }
  }
  if (t.cf) {
    std::vector<int32_t> info_h(2 * kInfoPerFactor);  // the factorisation's blocks, then the inverse's leaves
    double nrm[2];
    QTX_HIP(hipMemcpyAsync(info_h.data(), t.w.info, info_h.size() * sizeof(int32_t), hipMemcpyDeviceToHost, t.st));
    QTX_HIP(hipMemcpyAsync(nrm, t.w.scalars + 6, sizeof(nrm), hipMemcpyDeviceToHost, t.st));
    QTX_HIP(hipStreamSynchronize(t.st));
    bool ok = true;
    for (int32_t v : info_h) ok = ok && (v == 0);
    // nrm: |b' - T_d x|^2, |x|^2 of the result
    const double res = sqrt(nrm[0]), xn = sqrt(nrm[1]);
    const bool converged = std::isfinite(res) && std::isfinite(xn) && res <= kShiftAccept * t.lmax * xn;
    if (ok && converged) {
      hipLaunchKernelGGL(copy_f64_kernel, dim3(nblk(t.n, 256)), dim3(256), 0, t.st, t.w.x, t.w.y, t.n);
      QTX_LAUNCH_CHECK();
      t.path = 3;
    } else {  // T and y are intact: take the dsyevd route
      t.fallback = ok ? 7 : 6;
      int rc = snr_syevd(t, h);
      if (rc < 0) return rc;
      t.path = 2;
    }
  }
  if (t.minnorm) {
    int rc = launch_obar_t_y<TI>(t.st, (const TI*)io.O, io.mean, io.r, t.w.y, io.ns, io.np, io.step);
    if (rc) return rc;
  } else {
    hipLaunchKernelGGL(copy_f64_kernel, dim3(nblk(io.np, 256)), dim3(256), 0, t.st, t.w.y, io.step, io.np);
    QTX_LAUNCH_CHECK();
  }
  return QTX_OK;
}

static int check_task(const qtx_minsr_task& io) {
  QTX_REQUIRE(io.o_dtype == QTX_F32 || io.o_dtype == QTX_F64, "o_dtype must be QTX_F32 or QTX_F64");
  QTX_REQUIRE(io.ns > 0 && io.np > 0 && io.O && io.mean && io.ebar && io.step, "bad arguments");
  const int mode = base_mode(io.mode);
  QTX_REQUIRE(mode == QTX_SOLVE_CHOL_SHIFT || mode == QTX_SOLVE_EIGH_PINV || mode == QTX_SOLVE_EIGH_PINV_DIRECT,
              "unknown solver mode");
  QTX_REQUIRE((io.mode & ~(0xff | QTX_SOLVE_MINNORM | QTX_SOLVE_LSTSQ | QTX_SOLVE_SNR | QTX_SOLVE_BLAS_WS |
                            QTX_SOLVE_CHEB)) == 0 &&
                  !((io.mode & QTX_SOLVE_MINNORM) && (io.mode & QTX_SOLVE_LSTSQ)),
              "bad solver mode flags");
  QTX_REQUIRE(io.gram == QTX_GRAM_FP64 || io.gram == QTX_GRAM_FP32 || io.gram == QTX_GRAM_BF16X3,
              "unknown gram mode");
  QTX_REQUIRE((use_minnorm(io.ns, io.np, io.mode) ? io.ns : io.np) <= 131072, "matrix too large (n > 131072)");
  QTX_REQUIRE(!(io.tol_snr > kSnrMin) || mode == QTX_SOLVE_CHOL_SHIFT || (io.mode & QTX_SOLVE_SNR),
              "tol_snr > 0 needs QTX_SOLVE_SNR in the mode (and its workspace)");
  size_t need = ws_layout(io.ns, io.np, io.mode, io.gram, nullptr, nullptr);
  if (io.mode & QTX_SOLVE_BLAS_WS) need += 256;  // a non-empty rocBLAS scratch tail
  if (io.ws == nullptr || io.ws_bytes < need)
    return fail(QTX_EWORKSPACE, "workspace too small: need " + std::to_string(need) + " bytes");
  return QTX_OK;
}

// rocBLAS / rocSOLVER scratch of one solve: a device-memory size query (no
// kernels run, nothing is read or written) over every library call the solve
// can make, with its dimensions and with pointers into the caller's workspace
static int blas_query(rocblas_handle h, int64_t ns, int64_t np, int mode, SolveWs& w, size_t* bytes) {
  const bool mn = use_minnorm(ns, np, mode);
  const int64_t n = mn ? ns : np, nn = n * n;
  const rocblas_int ni = (rocblas_int)n;
  const int bm = base_mode(mode);
  const double one = 1.0, zero = 0.0, minus_one = -1.0;
  if (rocblas_start_device_memory_size_query(h) != rocblas_status_success)
    return fail(QTX_ESOLVER, "rocblas_start_device_memory_size_query failed");
  auto ok = [](rocblas_status s) {
    return s == rocblas_status_success || s == rocblas_status_size_increased || s == rocblas_status_size_unchanged;
  };
  bool good = true;
  if (!mn) {  // SR branch: S by row blocks of Obar, and the SNR products
    const rocblas_int npi = (rocblas_int)np, rows = (rocblas_int)obar_rows(ns, np);
    if (np > kGramTnMax)
      good &= ok(rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_transpose, npi, npi, rows, &one, w.obar,
                               npi, w.obar, npi, &zero, w.T, npi));
    if (mode & QTX_SOLVE_SNR)
      good &= ok(rocblas_dgemm(h, rocblas_operation_transpose, rocblas_operation_none, npi, rows, npi, &one, w.T, npi,
                               w.obar, npi, &zero, w.cbuf, npi));
  }
  if (bm == QTX_SOLVE_CHOL_SHIFT || bm == QTX_SOLVE_EIGH_PINV) {  // panels of the blocked Cholesky
    double* A = (bm == QTX_SOLVE_CHOL_SHIFT) ? w.T : w.T2;
    for (int64_t k = 0, kb; k < n; k += kb) {
      kb = chol_block(n - k, bm == QTX_SOLVE_CHOL_SHIFT ? 1 : 3);  // the smaller blocks: every call of either
      const int64_t m = n - k - kb;
      if (m == 0) break;
      double* Akk = A + k * n + k;
      good &= ok(rocblas_dtrsm(h, rocblas_side_right, rocblas_fill_lower, rocblas_operation_transpose,
                               rocblas_diagonal_non_unit, (rocblas_int)m, (rocblas_int)kb, &one, Akk, ni, Akk + kb,
                               ni));
      good &= ok(rocblas_dsyrk(h, rocblas_fill_lower, rocblas_operation_none, (rocblas_int)m, (rocblas_int)kb,
                               &minus_one, Akk + kb, ni, &one, A + (k + kb) * n + (k + kb), ni));
    }
  }
  if (bm != QTX_SOLVE_CHOL_SHIFT) {  // the dsyevd route (EIGH_PINV: its fallback)
    good &= ok(rocsolver_dsyevd(h, rocblas_evect_original, rocblas_fill_lower, ni, w.T, ni, w.D, w.E, w.info));
    good &= ok(rocblas_dgemv(h, rocblas_operation_transpose, ni, ni, &one, w.T, ni, w.y, 1, &zero, w.z, 1));
    good &= ok(rocblas_dgemv(h, rocblas_operation_none, ni, ni, &one, w.T, ni, w.z, 1, &zero, w.y, 1));
  }
  if (bm == QTX_SOLVE_EIGH_PINV) {  // small-cutoff and Chebyshev routes: inverse factor and its products
    good &= tri_inverse(h, nullptr, n, w.T2, n, w.T2 + nn, w.info, true) == QTX_OK;
    for (rocblas_operation op : {rocblas_operation_none, rocblas_operation_transpose})
      good &= ok(rocblas_dtrmv(h, rocblas_fill_lower, op, rocblas_diagonal_non_unit, ni, w.T2, ni, w.R, 1));
  }
  if (bm == QTX_SOLVE_EIGH_PINV) {  // partial fractions: T^2 and the refinement's triangular solves
    good &= ok(rocblas_dsyrk(h, rocblas_fill_lower, rocblas_operation_none, ni, ni, &one, w.T, ni, &zero, w.T2, ni));
    for (rocblas_operation op : {rocblas_operation_none, rocblas_operation_transpose})
      good &= ok(rocblas_dtrsm_strided_batched(h, rocblas_side_left, rocblas_fill_lower, op, rocblas_diagonal_non_unit,
                                               ni, 2, &one, w.T2, ni, nn, w.R, ni, 2 * n, 3));
  }
  size_t sz = 0;
  const rocblas_status st = rocblas_stop_device_memory_size_query(h, &sz);
  if (!good || st != rocblas_status_success) return fail(QTX_ESOLVER, "rocBLAS device memory size query failed");
  // at least 256 bytes: a zero-byte workspace would put the handle back under
  // rocBLAS's own memory management
  *bytes = std::max<size_t>(256, (sz + 255) & ~(size_t)255);
  return QTX_OK;
}

// QTX_SERIAL_FACTOR=1 runs the factorisations of different tasks one after
// another (default: they overlap on their streams)
static bool serial_factorisations() {
  static const bool v = [] {
    const char* e = getenv("QTX_SERIAL_FACTOR");
    return e && e[0] == '1';
  }();
  return v;
}

static int solve_many(qtx_minsr_task* tasks, int ntasks) {
  std::vector<Task> ts((size_t)ntasks);
  int first_rc = QTX_OK;
  std::string first_msg;
  auto note = [&](Task& t, int rc) {
    task_fail(t, rc);
    if (first_rc == QTX_OK) {
      first_rc = rc;
      first_msg = qtx_last_error();
    }
  };
  for (int i = 0; i < ntasks; ++i) {
    Task& t = ts[i];
    t.io = &tasks[i];
    t.io->status = QTX_OK;
    t.io->path = -1;
    t.io->fallback = 0;
    int rc = check_task(tasks[i]);
    if (rc) {
      note(t, rc);
      continue;
    }
    t.st = as_stream(tasks[i].stream);
    t.minnorm = use_minnorm(tasks[i].ns, tasks[i].np, tasks[i].mode);
    t.n = t.minnorm ? tasks[i].ns : tasks[i].np;
    const size_t own = ws_layout(tasks[i].ns, tasks[i].np, tasks[i].mode, tasks[i].gram, &t.w, (char*)tasks[i].ws);
    if (tasks[i].mode & QTX_SOLVE_BLAS_WS) {
      t.blas_ws = (char*)tasks[i].ws + own;
      t.blas_bytes = tasks[i].ws_bytes - own;
    }
  }
  rocblas_handle h = nullptr;
  for (int phase = 1; phase <= 3; ++phase) {
    for (Task& t : ts) {
      if (t.failed) continue;
      const bool user = (t.io->mode & QTX_SOLVE_BLAS_WS) != 0;
      int rc = get_blas(t.st, &h, t.blas_ws, t.blas_bytes, user);
      if (rc == QTX_OK) {
        rocblas_pointer_mode pm;
        rocblas_get_pointer_mode(h, &pm);
        rocblas_set_pointer_mode(h, rocblas_pointer_mode_host);
        const bool f32 = t.io->o_dtype == QTX_F32;
        if (phase == 1) rc = f32 ? phase1<float>(t, h) : phase1<double>(t, h);
        else if (phase == 2) rc = phase2(t, h);
        else rc = f32 ? phase3<float>(t, h) : phase3<double>(t, h);
        // factorisations of one task finish before the next task's start
        const bool factored = (phase == 1 && base_mode(t.io->mode) == QTX_SOLVE_CHOL_SHIFT) || (phase == 2 && t.pf);
        if (rc == QTX_OK && factored && ntasks > 1 && serial_factorisations())
          rc = hip_check(hipStreamSynchronize(t.st), "hipStreamSynchronize");
        rocblas_set_pointer_mode(h, pm);
      }
      if (rc) note(t, rc);
    }
  }
  for (Task& t : ts) {
    t.io->path = t.path;
    t.io->fallback = t.fallback;
  }
  if (ntasks > 0) {
    const Task& t = ts[ntasks - 1];
    g_last_path = t.failed ? -1 : t.path;
    g_last_lanczos = t.lanczos;
    g_last_lmax = t.lmax;
    g_last_fallback = t.fallback;
  }
  if (first_rc != QTX_OK) return fail(first_rc, first_msg);
  return QTX_OK;
}

extern "C" {

int qtx_colmean(void* stream, int o_dtype, const void* O, int64_t ns, int64_t np, double* mean) {
  QTX_REQUIRE(o_dtype == QTX_F32 || o_dtype == QTX_F64, "o_dtype must be QTX_F32 or QTX_F64");
  QTX_REQUIRE(ns > 0 && np > 0 && O && mean, "bad arguments");
  hipStream_t st = as_stream(stream);
  hipLaunchKernelGGL(fill_f64_kernel, dim3(nblk(np, 256)), dim3(256), 0, st, mean, np, 0.0);
  dim3 g;
  int lg;
  const int64_t rpc = colsum_rows(ns, np, g, lg);
  const double* none = nullptr;
  if (o_dtype == QTX_F32)
    hipLaunchKernelGGL((colsum_kernel<float, false>), g, dim3(256), 0, st, (const float*)O, none, none, none, ns, np,
                       rpc, lg, 0.0, mean);
  else
    hipLaunchKernelGGL((colsum_kernel<double, false>), g, dim3(256), 0, st, (const double*)O, none, none, none, ns, np,
                       rpc, lg, 0.0, mean);
  hipLaunchKernelGGL(scale_f64_kernel, dim3(nblk(np, 256)), dim3(256), 0, st, mean, np, 1.0 / (double)ns);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

int qtx_obar_matvec(void* stream, int o_dtype, const void* O, const double* mean, const double* r, int64_t ns,
                    int64_t np, double alpha, const double* v, double beta, double* y) {
  QTX_REQUIRE(o_dtype == QTX_F32 || o_dtype == QTX_F64, "o_dtype must be QTX_F32 or QTX_F64");
  QTX_REQUIRE(ns > 0 && np > 0 && O && mean && v && y, "bad arguments");
  hipStream_t st = as_stream(stream);
  dim3 g(nblk(ns, 256 / WAVE));
  if (o_dtype == QTX_F32)
    hipLaunchKernelGGL(obar_matvec_kernel<float>, g, dim3(256), 0, st, (const float*)O, mean, r, ns, np,
                       1.0 / (double)ns, alpha, v, beta, y);
  else
    hipLaunchKernelGGL(obar_matvec_kernel<double>, g, dim3(256), 0, st, (const double*)O, mean, r, ns, np,
                       1.0 / (double)ns, alpha, v, beta, y);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

int qtx_scale_columns(void* stream, int o_dtype, void* O, double* mean, int64_t ns, int64_t np, const double* d) {
  QTX_REQUIRE(o_dtype == QTX_F32 || o_dtype == QTX_F64, "o_dtype must be QTX_F32 or QTX_F64");
  QTX_REQUIRE(ns > 0 && np > 0 && O && d, "bad arguments");
  hipStream_t st = as_stream(stream);
  const unsigned grid = (unsigned)std::min<int64_t>((ns * np + 255) / 256, kGridCap);
  if (o_dtype == QTX_F32)
    hipLaunchKernelGGL(scale_columns_kernel<float>, dim3(grid), dim3(256), 0, st, (float*)O, ns, np, d);
  else
    hipLaunchKernelGGL(scale_columns_kernel<double>, dim3(grid), dim3(256), 0, st, (double*)O, ns, np, d);
  if (mean) hipLaunchKernelGGL(mul_f64_kernel, dim3(nblk(np, 256)), dim3(256), 0, st, mean, d, np);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

int qtx_ebar(void* stream, const double* eloc, const double* r, int64_t ns, double* ebar, double* out2) {
  QTX_REQUIRE(ns > 0 && eloc && ebar && out2, "bad arguments");
  hipLaunchKernelGGL(ebar_kernel, dim3(1), dim3(1024), 0, as_stream(stream), eloc, r, ns, ebar, out2);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

size_t qtx_minsr_ws_bytes(int64_t ns, int64_t np, int mode, int gram) {
  if (ns <= 0 || np <= 0) return 0;
  return ws_layout(ns, np, mode, gram, nullptr, nullptr);
}

int qtx_minsr_solve(void* stream, int o_dtype, const void* O, const double* mean, const double* r,
                    const double* ebar, int64_t ns, int64_t np, int mode, int gram, double rshift, double ashift,
                    double rtol, double atol, double* step, void* ws, size_t ws_bytes) {
  qtx_minsr_task task{};
  task.stream = stream;
  task.o_dtype = o_dtype;
  task.mode = mode;
  task.gram = gram;
  task.O = O;
  task.mean = mean;
  task.r = r;
  task.ebar = ebar;
  task.ns = ns;
  task.np = np;
  task.rshift = rshift;
  task.ashift = ashift;
  task.rtol = rtol;
  task.atol = atol;
  task.step = step;
  task.ws = ws;
  task.ws_bytes = ws_bytes;
  g_last_path = -1;
  g_last_lanczos = 0;
  g_last_lmax = 0.0;
  g_last_fallback = 0;
  return solve_many(&task, 1);
}

int qtx_minsr_solve_many(qtx_minsr_task* tasks, int32_t ntasks) {
  QTX_REQUIRE(ntasks >= 0 && (ntasks == 0 || tasks != nullptr), "bad task array");
  return solve_many(tasks, ntasks);
}

int qtx_minsr_last_path(int* path, int* lanczos_steps, double* lambda_max, int* fallback) {
  QTX_REQUIRE(path && lanczos_steps && lambda_max, "bad arguments");
  if (fallback) *fallback = g_last_fallback;
  *path = g_last_path;
  *lanczos_steps = g_last_lanczos;
  *lambda_max = g_last_lmax;
  return QTX_OK;
}

size_t qtx_gram_ws_bytes(int64_t ns, int64_t np, int gram) {
  if (ns <= 0 || np <= 0 || gram != QTX_GRAM_BF16X3 || ns >= np) return 0;
  return g3_bytes(ns, np);
}

int qtx_gram(void* stream, int o_dtype, const void* O, const double* mean, const double* r, int64_t ns,
             int64_t np, int gram, double* T, void* ws, size_t ws_bytes) {
  QTX_REQUIRE(o_dtype == QTX_F32 || o_dtype == QTX_F64, "o_dtype must be QTX_F32 or QTX_F64");
  QTX_REQUIRE(ns > 0 && np > 0 && O && mean && T, "bad arguments");
  QTX_REQUIRE(gram == QTX_GRAM_FP64 || gram == QTX_GRAM_FP32 || gram == QTX_GRAM_BF16X3, "unknown gram mode");
  const size_t need = qtx_gram_ws_bytes(ns, np, gram);
  if (need > 0 && (ws == nullptr || ws_bytes < need))
    return fail(QTX_EWORKSPACE, "workspace too small: need " + std::to_string(need) + " bytes");
  hipStream_t st = as_stream(stream);
  if (ns < np) {
    if (o_dtype == QTX_F32) return launch_gram_nt<float>(st, gram, (const float*)O, mean, r, ns, np, T, ws);
    return launch_gram_nt<double>(st, gram, (const double*)O, mean, r, ns, np, T, ws);
  }
  if (o_dtype == QTX_F32) return launch_gram_tn<float>(st, (const float*)O, mean, r, ns, np, T);
  return launch_gram_tn<double>(st, (const double*)O, mean, r, ns, np, T);
}

int qtx_apply_update(void* stream, int dtype, void* theta, const double* step, double lr, int64_t np,
                     int32_t* applied) {
  QTX_REQUIRE(dtype == QTX_F32 || dtype == QTX_F64, "dtype must be QTX_F32 or QTX_F64");
  QTX_REQUIRE(np > 0 && theta && step && applied, "bad arguments");
  hipStream_t st = as_stream(stream);
  hipLaunchKernelGGL(fill_i32_kernel, dim3(1), dim3(64), 0, st, applied, (int64_t)1, 1);
  hipLaunchKernelGGL(finite_check_kernel<double>, dim3(nblk(np, 256)), dim3(256), 0, st, step, np, applied);
  if (dtype == QTX_F32)
    hipLaunchKernelGGL(apply_update_kernel<float>, dim3(nblk(np, 256)), dim3(256), 0, st, (float*)theta, step, lr,
                       np, applied);
  else
    hipLaunchKernelGGL(apply_update_kernel<double>, dim3(nblk(np, 256)), dim3(256), 0, st, (double*)theta, step,
                       lr, np, applied);
  QTX_LAUNCH_CHECK();
  return QTX_OK;
}

int qtx_minsr_blas_ws_bytes(void* stream, int64_t ns, int64_t np, int mode, int gram, void* ws, size_t ws_bytes,
                            size_t* bytes) {
  QTX_REQUIRE(ns > 0 && np > 0 && bytes, "bad arguments");
  const int bm = base_mode(mode);
  QTX_REQUIRE(bm == QTX_SOLVE_CHOL_SHIFT || bm == QTX_SOLVE_EIGH_PINV || bm == QTX_SOLVE_EIGH_PINV_DIRECT,
              "unknown solver mode");
  const size_t own = ws_layout(ns, np, mode, gram, nullptr, nullptr);
  if (ws == nullptr || ws_bytes < own)
    return fail(QTX_EWORKSPACE, "workspace too small: need " + std::to_string(own) + " bytes");
  SolveWs w{};
  ws_layout(ns, np, mode, gram, &w, (char*)ws);
  rocblas_handle h = nullptr;
  int rc = get_blas(as_stream(stream), &h, nullptr, 0, true);
  if (rc) return rc;
  rocblas_pointer_mode pm;
  rocblas_get_pointer_mode(h, &pm);
  rocblas_set_pointer_mode(h, rocblas_pointer_mode_host);
  rc = blas_query(h, ns, np, mode, w, bytes);
  rocblas_set_pointer_mode(h, pm);
  return rc;
}

int qtx_minsr_solve_snr(void* stream, int o_dtype, const void* O, const double* mean, const double* r,
                        const double* ebar, int64_t ns, int64_t np, int mode, int gram, double rtol, double atol,
                        double tol_snr, double* step, void* ws, size_t ws_bytes) {
  QTX_REQUIRE(base_mode(mode) == QTX_SOLVE_EIGH_PINV || base_mode(mode) == QTX_SOLVE_EIGH_PINV_DIRECT,
              "SNR truncation applies to the EIGH_PINV modes");
  QTX_REQUIRE(tol_snr >= 0.0, "tol_snr must be >= 0");
  qtx_minsr_task task{};
  task.stream = stream;
  task.o_dtype = o_dtype;
  task.mode = mode | QTX_SOLVE_SNR;
  task.gram = gram;
  task.O = O;
  task.mean = mean;
  task.r = r;
  task.ebar = ebar;
  task.ns = ns;
  task.np = np;
  task.rtol = rtol;
  task.atol = atol;
  task.tol_snr = tol_snr;
  task.step = step;
  task.ws = ws;
  task.ws_bytes = ws_bytes;
  g_last_path = -1;
  g_last_lanczos = 0;
  g_last_lmax = 0.0;
  g_last_fallback = 0;
  return solve_many(&task, 1);
}

// the MinSR-branch layout of an n x n problem: T, y, z, D, E, scalars and var2
static constexpr int kPinvEigMode = QTX_SOLVE_EIGH_PINV_DIRECT | QTX_SOLVE_MINNORM | QTX_SOLVE_SNR;

size_t qtx_pinv_eig_ws_bytes(int64_t n) {
  if (n <= 0) return 0;
  return ws_layout(n, n, kPinvEigMode, QTX_GRAM_FP64, nullptr, nullptr);
}

int qtx_pinv_eig(void* stream, const double* T, int64_t n, const double* b, double rtol, double atol, double tol_snr,
                 double* x, void* ws, size_t ws_bytes) {
  QTX_REQUIRE(n > 0 && T && b && x, "bad arguments");
  QTX_REQUIRE(n <= 131072, "matrix too large (n > 131072)");
  QTX_REQUIRE(rtol >= 0.0 && atol >= 0.0 && tol_snr >= 0.0, "tolerances must be >= 0");
  const size_t need = qtx_pinv_eig_ws_bytes(n);
  if (ws == nullptr || ws_bytes < need)
    return fail(QTX_EWORKSPACE, "workspace too small: need " + std::to_string(need) + " bytes");
  hipStream_t st = as_stream(stream);
  SolveWs w{};
  ws_layout(n, n, kPinvEigMode, QTX_GRAM_FP64, &w, (char*)ws);
  QTX_HIP(hipMemcpyAsync(w.T, T, (size_t)n * n * 8, hipMemcpyDeviceToDevice, st));
  QTX_HIP(hipMemcpyAsync(w.y, b, (size_t)n * 8, hipMemcpyDeviceToDevice, st));
  rocblas_handle h = nullptr;
  int rc = get_blas(st, &h);
  if (rc) return rc;
  rocblas_pointer_mode pm;
  rocblas_get_pointer_mode(h, &pm);
  rocblas_set_pointer_mode(h, rocblas_pointer_mode_host);
  rc = pinv_syevd(st, h, n, rtol, atol, w, tol_snr, nullptr);
  rocblas_set_pointer_mode(h, pm);
  if (rc < 0) return rc;
  QTX_HIP(hipMemcpyAsync(x, w.y, (size_t)n * 8, hipMemcpyDeviceToDevice, st));
  return QTX_OK;
}

}  // extern "C"
