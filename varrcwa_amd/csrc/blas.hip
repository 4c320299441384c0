// Complex128 dense kernels for gfx950: FP64-MFMA ZGEMM (strided batches)
// and the elementwise matrix kernels used between the factorizations.
//
// ZGEMM tiles: 64x64 output per workgroup (8 wavefronts by default; a 4-wave variant
// selectable), or 32x32 where few tiles would leave CUs idle, from v_mfma_f64_16x16x4f64
// blocks, K staged through LDS in chunks of 16 (32) complex values, real and imaginary planes
// kept separate so that one complex multiply-add is four real MFMAs (standard 4M product, no
// 3M/Gauss trick).
#include "vrc_common.hpp"
#include "vrc_internal.hpp"

namespace vrc {

constexpr int GT_M = 64, GT_N = 64, GT_K = 16, GT_THREADS = 256;

template <int OPA, int OPB>
__device__ __forceinline__ void zgemm_tile(int m, int n, int k, cd alpha, const cd* __restrict__ A, long lda,
                                           const cd* __restrict__ B, long ldb, cd beta, cd* __restrict__ C,
                                           long ldc, int tm, int tn) {
  __shared__ double As_re[GT_K][GT_M + 1];
  __shared__ double As_im[GT_K][GT_M + 1];
  __shared__ double Bs_re[GT_K][GT_N + 1];
  __shared__ double Bs_im[GT_K][GT_N + 1];

  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  const int row0 = tm * GT_M, col0 = tn * GT_N;

  d4 accR[2][2], accI[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      accR[i][j] = d4{0.0, 0.0, 0.0, 0.0};
      accI[i][j] = d4{0.0, 0.0, 0.0, 0.0};
    }

  // op(A) tile (GT_M x GT_K) and op(B) tile (GT_K x GT_N), 4 elements each per thread;
  // the next K chunk is fetched into registers while the current one is multiplied
  cd pa[4], pb[4];
  auto fetch = [&](int kk) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      cd v = mk(0.0, 0.0);
      if (OPA == OP_N) {
        const int gr = row0 + (t & 63), gc = kk + (t >> 6) + 4 * i;
        if (gr < m && gc < k) v = A[gr + (long)gc * lda];
      } else {
        const int gr = row0 + (t >> 4) + 16 * i, gc = kk + (t & 15);
        if (gr < m && gc < k) v = A[gc + (long)gr * lda];
        if (OPA == OP_C) v.y = -v.y;
      }
      pa[i] = v;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      cd v = mk(0.0, 0.0);
      if (OPB == OP_N) {
        const int gc = kk + (t & 15), gj = col0 + (t >> 4) + 16 * i;
        if (gc < k && gj < n) v = B[gc + (long)gj * ldb];
      } else {
        const int gc = kk + (t >> 6) + 4 * i, gj = col0 + (t & 63);
        if (gc < k && gj < n) v = B[gj + (long)gc * ldb];
        if (OPB == OP_C) v.y = -v.y;
      }
      pb[i] = v;
    }
  };
  fetch(0);
  for (int kk = 0; kk < k; kk += GT_K) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (OPA == OP_N) {
        As_re[(t >> 6) + 4 * i][t & 63] = pa[i].x;
        As_im[(t >> 6) + 4 * i][t & 63] = pa[i].y;
      } else {
        As_re[t & 15][(t >> 4) + 16 * i] = pa[i].x;
        As_im[t & 15][(t >> 4) + 16 * i] = pa[i].y;
      }
      if (OPB == OP_N) {
        Bs_re[t & 15][(t >> 4) + 16 * i] = pb[i].x;
        Bs_im[t & 15][(t >> 4) + 16 * i] = pb[i].y;
      } else {
        Bs_re[(t >> 6) + 4 * i][t & 63] = pb[i].x;
        Bs_im[(t >> 6) + 4 * i][t & 63] = pb[i].y;
      }
    }
    __syncthreads();
    if (kk + GT_K < k) fetch(kk + GT_K);
#pragma unroll
    for (int s = 0; s < GT_K / 4; ++s) {
      const int kr = s * 4 + (lane >> 4);
      double ar[2], ai[2], nai[2], br[2], bi[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        ar[b] = As_re[kr][wr * 32 + b * 16 + (lane & 15)];
        ai[b] = As_im[kr][wr * 32 + b * 16 + (lane & 15)];
        nai[b] = -ai[b];
        br[b] = Bs_re[kr][wc * 32 + b * 16 + (lane & 15)];
        bi[b] = Bs_im[kr][wc * 32 + b * 16 + (lane & 15)];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], br[j], accR[i][j], 0, 0, 0);
          accR[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(nai[i], bi[j], accR[i][j], 0, 0, 0);
          accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], bi[j], accI[i][j], 0, 0, 0);
          accI[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[i], br[j], accI[i][j], 0, 0, 0);
        }
    }
    __syncthreads();
  }

  // ---- epilogue: D layout of v_mfma_f64_16x16x4f64: register r of a lane holds row lane/16 + 4*r,
  // column lane%16 (established on gfx950 against a reference product)
  const bool beta0 = (beta.x == 0.0 && beta.y == 0.0);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int gc = col0 + wc * 32 + j * 16 + (lane & 15);
      if (gc >= n) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gr = row0 + wr * 32 + i * 16 + (lane >> 4) + 4 * r;
        if (gr >= m) continue;
        cd acc = mk(accR[i][j][r], accI[i][j][r]);
        cd out = cmul(alpha, acc);
        cd* cp = C + gr + (long)gc * ldc;
        if (!beta0) out = cadd(out, cmul(beta, *cp));
        *cp = out;
      }
    }
}

// The 64x64 tile on eight waves (512 threads): wave w owns rows 32*(w>>2) .. +32 and
// columns 16*(w&3) .. +16 (2x1 blocks); staging as above, 2 elements per thread.
template <int OPA, int OPB>
__device__ __forceinline__ void zgemm_tile8(int m, int n, int k, cd alpha, const cd* __restrict__ A, long lda,
                                            const cd* __restrict__ B, long ldb, cd beta, cd* __restrict__ C,
                                            long ldc, int tm, int tn) {
  __shared__ double As_re[GT_K][GT_M + 1];
  __shared__ double As_im[GT_K][GT_M + 1];
  __shared__ double Bs_re[GT_K][GT_N + 1];
  __shared__ double Bs_im[GT_K][GT_N + 1];
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int wr = wave >> 2, wc = wave & 3;
  const int row0 = tm * GT_M, col0 = tn * GT_N;
  d4 accR[2], accI[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    accR[i] = d4{0.0, 0.0, 0.0, 0.0};
    accI[i] = d4{0.0, 0.0, 0.0, 0.0};
  }
  // element q of this thread: A (row t&63, k (t>>6) + 8q) or (row (t>>4) + 32q, k t&15);
  // B (k t&15, col (t>>4) + 32q) or (k (t>>6) + 8q, col t&63)
  cd pa[2], pb[2];
  auto fetch = [&](int kk) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      cd v = mk(0.0, 0.0);
      if (OPA == OP_N) {
        const int gr = row0 + (t & 63), gc = kk + (t >> 6) + 8 * i;
        if (gr < m && gc < k) v = A[gr + (long)gc * lda];
      } else {
        const int gr = row0 + (t >> 4) + 32 * i, gc = kk + (t & 15);
        if (gr < m && gc < k) v = A[gc + (long)gr * lda];
        if (OPA == OP_C) v.y = -v.y;
      }
      pa[i] = v;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      cd v = mk(0.0, 0.0);
      if (OPB == OP_N) {
        const int gc = kk + (t & 15), gj = col0 + (t >> 4) + 32 * i;
        if (gc < k && gj < n) v = B[gc + (long)gj * ldb];
      } else {
        const int gc = kk + (t >> 6) + 8 * i, gj = col0 + (t & 63);
        if (gc < k && gj < n) v = B[gj + (long)gc * ldb];
        if (OPB == OP_C) v.y = -v.y;
      }
      pb[i] = v;
    }
  };
  fetch(0);
  for (int kk = 0; kk < k; kk += GT_K) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (OPA == OP_N) {
        As_re[(t >> 6) + 8 * i][t & 63] = pa[i].x;
        As_im[(t >> 6) + 8 * i][t & 63] = pa[i].y;
      } else {
        As_re[t & 15][(t >> 4) + 32 * i] = pa[i].x;
        As_im[t & 15][(t >> 4) + 32 * i] = pa[i].y;
      }
      if (OPB == OP_N) {
        Bs_re[t & 15][(t >> 4) + 32 * i] = pb[i].x;
        Bs_im[t & 15][(t >> 4) + 32 * i] = pb[i].y;
      } else {
        Bs_re[(t >> 6) + 8 * i][t & 63] = pb[i].x;
        Bs_im[(t >> 6) + 8 * i][t & 63] = pb[i].y;
      }
    }
    __syncthreads();
    if (kk + GT_K < k) fetch(kk + GT_K);
#pragma unroll
    for (int s = 0; s < GT_K / 4; ++s) {
      const int kr = s * 4 + (lane >> 4);
      double ar[2], ai[2], nai[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        ar[b] = As_re[kr][wr * 32 + b * 16 + (lane & 15)];
        ai[b] = As_im[kr][wr * 32 + b * 16 + (lane & 15)];
        nai[b] = -ai[b];
      }
      const double br = Bs_re[kr][wc * 16 + (lane & 15)], bi = Bs_im[kr][wc * 16 + (lane & 15)];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        accR[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], br, accR[i], 0, 0, 0);
        accR[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(nai[i], bi, accR[i], 0, 0, 0);
        accI[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], bi, accI[i], 0, 0, 0);
        accI[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[i], br, accI[i], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  const bool beta0 = (beta.x == 0.0 && beta.y == 0.0);
  const int gc = col0 + wc * 16 + (lane & 15);
  if (gc >= n) return;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int gr = row0 + wr * 32 + i * 16 + (lane >> 4) + 4 * r;
      if (gr >= m) continue;
      cd out = cmul(alpha, mk(accR[i][r], accI[i][r]));
      cd* cp = C + gr + (long)gc * ldc;
      if (!beta0) out = cadd(out, cmul(beta, *cp));
      *cp = out;
    }
}

// 32x32 output per 256-thread workgroup (four waves, one 16x16 block each) with K in chunks of
// 32, for products whose larger tiles would leave most CUs without a workgroup (single
// matrices and short right-hand sides): latency-bound there, so the tile is small and a barrier
// covers 32 k. Every element is summed in the order of the 64x64 tile, so the two agree to
// the last bit.
constexpr int GS_T = 32, GS_K = 32, GS_THREADS = 256;

template <int OPA, int OPB>
__device__ __forceinline__ void zgemm_tile32(int m, int n, int k, cd alpha, const cd* __restrict__ A, long lda,
                                             const cd* __restrict__ B, long ldb, cd beta, cd* __restrict__ C, long ldc,
                                             int tm, int tn) {
  __shared__ double As_re[GS_K][GS_T + 1];
  __shared__ double As_im[GS_K][GS_T + 1];
  __shared__ double Bs_re[GS_K][GS_T + 1];
  __shared__ double Bs_im[GS_K][GS_T + 1];
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = t >> 6;
  const int wr = wave >> 1, wc = wave & 1;
  const int row0 = tm * GS_T, col0 = tn * GS_T;
  const bool live = __builtin_amdgcn_readfirstlane(row0 + wr * 16 < m && col0 + wc * 16 < n);
  d4 accR = d4{0.0, 0.0, 0.0, 0.0}, accI = accR;
  // element q of this thread: (x, y) = (t & 31, (t >> 5) + 8 q), x along the operand's columns
  const int x = t & 31, y = t >> 5;
  cd pa[4], pb[4];
  auto fetch = [&](int kk) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int yy = y + 8 * q;
      cd v = mk(0.0, 0.0);
      if (OPA == OP_N) {
        if (row0 + x < m && kk + yy < k) v = A[(row0 + x) + (long)(kk + yy) * lda];
      } else {
        if (row0 + yy < m && kk + x < k) v = A[(kk + x) + (long)(row0 + yy) * lda];
        if (OPA == OP_C) v.y = -v.y;
      }
      pa[q] = v;
      v = mk(0.0, 0.0);
      if (OPB == OP_N) {
        if (kk + x < k && col0 + yy < n) v = B[(kk + x) + (long)(col0 + yy) * ldb];
      } else {
        if (kk + yy < k && col0 + x < n) v = B[(col0 + x) + (long)(kk + yy) * ldb];
        if (OPB == OP_C) v.y = -v.y;
      }
      pb[q] = v;
    }
  };
  fetch(0);
  for (int kk = 0; kk < k; kk += GS_K) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int yy = y + 8 * q;
      (OPA == OP_N ? As_re[yy][x] : As_re[x][yy]) = pa[q].x;
      (OPA == OP_N ? As_im[yy][x] : As_im[x][yy]) = pa[q].y;
      (OPB == OP_N ? Bs_re[x][yy] : Bs_re[yy][x]) = pb[q].x;
      (OPB == OP_N ? Bs_im[x][yy] : Bs_im[yy][x]) = pb[q].y;
    }
    __syncthreads();
    if (kk + GS_K < k) fetch(kk + GS_K);
    if (live) {
#pragma unroll
      for (int s = 0; s < GS_K / 4; ++s) {
        const int kr = s * 4 + (lane >> 4);
        const double ar = As_re[kr][wr * 16 + (lane & 15)], ai = As_im[kr][wr * 16 + (lane & 15)];
        const double br = Bs_re[kr][wc * 16 + (lane & 15)], bi = Bs_im[kr][wc * 16 + (lane & 15)];
        accR = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, br, accR, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, bi, accI, 0, 0, 0);
        accR = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai, bi, accR, 0, 0, 0);
        accI = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, br, accI, 0, 0, 0);
      }
    }
    __syncthreads();
  }
  const bool beta0 = (beta.x == 0.0 && beta.y == 0.0);
  const int gc = col0 + wc * 16 + (lane & 15);
  if (gc >= n) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int gr = row0 + wr * 16 + (lane >> 4) + 4 * r;
    if (gr >= m) continue;
    cd out = cmul(alpha, mk(accR[r], accI[r]));
    cd* cp = C + gr + (long)gc * ldc;
    if (!beta0) out = cadd(out, cmul(beta, *cp));
    *cp = out;
  }
}

// Scale-only path for k == 0 (C = beta*C).
__device__ __forceinline__ void scale_tile(int m, int n, cd beta, cd* C, long ldc, int tm, int tn) {
  const bool beta0 = (beta.x == 0.0 && beta.y == 0.0);
  for (int e = threadIdx.x; e < GT_M * GT_N; e += GT_THREADS) {
    int r = e % GT_M, c = e / GT_M;
    int gr = tm * GT_M + r, gc = tn * GT_N + c;
    if (gr < m && gc < n) {
      cd* p = C + gr + (long)gc * ldc;
      *p = beta0 ? mk(0.0, 0.0) : cmul(beta, *p);
    }
  }
}

template <int OPA, int OPB>
__global__ __launch_bounds__(GT_THREADS) void zgemm_strided_kernel(int m, int n, int k, cd alpha, const cd* A,
                                                                   long lda, long sA, const cd* B, long ldb,
                                                                   long sB, cd beta, cd* C, long ldc, long sC) {
  const int tm = blockIdx.x, tn = blockIdx.y;
  const long b = blockIdx.z;
  if (k <= 0) {
    scale_tile(m, n, beta, C + b * sC, ldc, tm, tn);
    return;
  }
  zgemm_tile<OPA, OPB>(m, n, k, alpha, A + b * sA, lda, B + b * sB, ldb, beta, C + b * sC, ldc, tm, tn);
}

// Transposed operands: six waves per SIMD (80 registers) measured 63.2 TFLOP/s at 250 x 882^3 (C,
// N) against 59.9; plain operands run best as the compiler allocates them (64.8 against 63.4).
template <int OPA, int OPB>
__global__ __launch_bounds__(512, OPA == OP_N && OPB == OP_N ? 1 : 6) void zgemm_strided8_kernel(
    int m, int n, int k, cd alpha, const cd* A, long lda, long sA, const cd* B, long ldb, long sB, cd beta, cd* C,
    long ldc, long sC) {
  const int tm = blockIdx.x, tn = blockIdx.y;
  const long b = blockIdx.z;
  zgemm_tile8<OPA, OPB>(m, n, k, alpha, A + b * sA, lda, B + b * sB, ldb, beta, C + b * sC, ldc, tm, tn);
}

template <int OPA, int OPB>
__global__ __launch_bounds__(GS_THREADS) void zgemm_small_kernel(int m, int n, int k, cd alpha, const cd* A, long lda,
                                                                long sA, const cd* B, long ldb, long sB, cd beta,
                                                                cd* C, long ldc, long sC) {
  const int tm = blockIdx.x, tn = blockIdx.y;
  const long b = blockIdx.z;
  zgemm_tile32<OPA, OPB>(m, n, k, alpha, A + b * sA, lda, B + b * sB, ldb, beta, C + b * sC, ldc, tm, tn);
}

static int g_small_waves = 8;   // wavefronts of the 64x64-tile kernel (4 or 8)
void zgemm_set_small_waves(int w) { g_small_waves = w == 8 ? 8 : 4; }
int zgemm_get_small_waves() { return g_small_waves; }

// 32x32 instead of 64x64 tiles? A 64x64 workgroup takes about 0.14 us per unit of k, a 32x32 one
// 0.054 us, one per CU at a time either way while workgroups are few, so the smaller tile wins
// while its rounds over the 256 CUs cost less (single matrices and short right-hand sides;
// us with 64 / 32: 162^3 26 / 12, 450^3 65 / 27, 882^3 126 / 141, 64 x 484 x 64 12 / 6, 16
// products of 242^3 43 / 54), or where 64 fits the edges so badly that 32 saves more than an eighth
// of the tiles' area (37 and 129 are the costs of one tile with the chip full; 256 products
// 81 x 81 x 128: 74 / 56). Tiles of 128x64 and 128x128 are gone: slower than 64x64 with plain
// operands at every size measured (N = 242 .. 1250, batches of 1 .. 2000; 250 products of 882^3:
// 22.2 ms against 21.3) and with transposed ones at most (N = 128 .. 882, batches of 8 .. 150: 0.94 to
// 2.7 times their speed; below 1 only where 200 to 256 tiles of 128x128 made one full round).
static bool zgemm_use_32(int m, int n, int k, int batch) {
  const long n64 = (long)cdiv_up(m, GT_M) * cdiv_up(n, GT_N) * batch;
  const long n32 = (long)cdiv_up(m, GS_T) * cdiv_up(n, GS_T) * batch;
  const long r64 = (n64 + 255) / 256, r32 = (n32 + 255) / 256;
  if (k <= 16) return r32 == 1;  // half a chunk of the 32x32 kernel
  if (r32 <= 8) return 27 * r32 < 70 * r64;
  return 37 * n32 < 129 * n64;
}

void zgemm_strided(hipStream_t s, int opA, int opB, int m, int n, int k, cd alpha, const cd* A, long lda,
                   long sA, const cd* B, long ldb, long sB, cd beta, cd* C, long ldc, long sC, int batch) {
  if (m <= 0 || n <= 0 || batch <= 0) return;
  if (k > 0 && zgemm_use_32(m, n, k, batch)) {
    dim3 grid(cdiv_up(m, GS_T), cdiv_up(n, GS_T), batch);
#define VRC_S32(OA, OB) \
  zgemm_small_kernel<OA, OB><<<grid, GS_THREADS, 0, s>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC)
    switch (opA * 3 + opB) {
      case 0: VRC_S32(OP_N, OP_N); break;
      case 1: VRC_S32(OP_N, OP_T); break;
      case 2: VRC_S32(OP_N, OP_C); break;
      case 3: VRC_S32(OP_T, OP_N); break;
      case 4: VRC_S32(OP_T, OP_T); break;
      case 5: VRC_S32(OP_T, OP_C); break;
      case 6: VRC_S32(OP_C, OP_N); break;
      case 7: VRC_S32(OP_C, OP_T); break;
      default: VRC_S32(OP_C, OP_C); break;
    }
#undef VRC_S32
    launch_check("zgemm_small");
    return;
  }
  dim3 grid(cdiv_up(m, GT_M), cdiv_up(n, GT_N), batch);
  if (g_small_waves == 8 && k > 0) {
#define VRC_S8(OA, OB) \
  zgemm_strided8_kernel<OA, OB><<<grid, 512, 0, s>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC)
    switch (opA * 3 + opB) {
      case 0: VRC_S8(OP_N, OP_N); break;
      case 1: VRC_S8(OP_N, OP_T); break;
      case 2: VRC_S8(OP_N, OP_C); break;
      case 3: VRC_S8(OP_T, OP_N); break;
      case 4: VRC_S8(OP_T, OP_T); break;
      case 5: VRC_S8(OP_T, OP_C); break;
      case 6: VRC_S8(OP_C, OP_N); break;
      case 7: VRC_S8(OP_C, OP_T); break;
      default: VRC_S8(OP_C, OP_C); break;
    }
#undef VRC_S8
    launch_check("zgemm_strided8");
    return;
  }
  switch (opA * 3 + opB) {
    case 0: zgemm_strided_kernel<OP_N, OP_N><<<grid, GT_THREADS, 0, s>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC); break;
    case 1: zgemm_strided_kernel<OP_N, OP_T><<<grid, GT_THREADS, 0, s>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC); break;
    case 2: zgemm_strided_kernel<OP_N, OP_C><<<grid, GT_THREADS, 0, s>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC); break;
    case 3: zgemm_strided_kernel<OP_T, OP_N><<<grid, GT_THREADS, 0, s>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC); break;
    case 4: zgemm_strided_kernel<OP_T, OP_T><<<grid, GT_THREADS, 0, s>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC); break;
    case 5: zgemm_strided_kernel<OP_T, OP_C><<<grid, GT_THREADS, 0, s>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC); break;
    case 6: zgemm_strided_kernel<OP_C, OP_N><<<grid, GT_THREADS, 0, s>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC); break;
    case 7: zgemm_strided_kernel<OP_C, OP_T><<<grid, GT_THREADS, 0, s>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC); break;
    default: zgemm_strided_kernel<OP_C, OP_C><<<grid, GT_THREADS, 0, s>>>(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC); break;
  }
  launch_check("zgemm_strided");
}

// ============================================================ elementwise kernels
// All take a strided batch of m x n column-major matrices.

__global__ void geam_kernel(int m, int n, cd a, const cd* A, long lda, long sA, cd b, const cd* B, long ldb,
                            long sB, cd* C, long ldc, long sC) {
  const long bz = blockIdx.z;
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (r >= m) return;
  cd v = cmul(a, A[bz * sA + r + (long)c * lda]);
  if (B) v = cadd(v, cmul(b, B[bz * sB + r + (long)c * ldb]));
  C[bz * sC + r + (long)c * ldc] = v;
}

void zgeam(hipStream_t s, int m, int n, cd a, const cd* A, long lda, long sA, cd b, const cd* B, long ldb, long sB,
           cd* C, long ldc, long sC, int batch) {
  if (m <= 0 || n <= 0 || batch <= 0) return;
  dim3 grid(cdiv_up(m, 256), n, batch);
  geam_kernel<<<grid, 256, 0, s>>>(m, n, a, A, lda, sA, b, B, ldb, sB, C, ldc, sC);
  launch_check("zgeam");
}

__global__ void set_ident_kernel(int m, int n, cd diag, cd off, cd* C, long ldc, long sC) {
  const long bz = blockIdx.z;
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (r >= m) return;
  C[bz * sC + r + (long)c * ldc] = (r == c) ? diag : off;
}

void zset(hipStream_t s, int m, int n, cd diag, cd off, cd* C, long ldc, long sC, int batch) {
  if (m <= 0 || n <= 0 || batch <= 0) return;
  dim3 grid(cdiv_up(m, 256), n, batch);
  set_ident_kernel<<<grid, 256, 0, s>>>(m, n, diag, off, C, ldc, sC);
  launch_check("zset");
}

__global__ void add_diag_kernel(int n, cd v, const cd* vec, long svec, cd* C, long ldc, long sC) {
  const long bz = blockIdx.y;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  cd add = vec ? cmul(v, vec[bz * svec + i]) : v;
  cd* p = C + bz * sC + i + (long)i * ldc;
  *p = cadd(*p, add);
}

void zadd_diag(hipStream_t s, int n, cd v, const cd* vec, long svec, cd* C, long ldc, long sC, int batch) {
  if (n <= 0 || batch <= 0) return;
  dim3 grid(cdiv_up(n, 256), batch);
  add_diag_kernel<<<grid, 256, 0, s>>>(n, v, vec, svec, C, ldc, sC);
  launch_check("zadd_diag");
}

// C = diag(left) * A * diag(right) (either vector may be null); in place allowed.
__global__ void dscale_kernel(int m, int n, const cd* left, long sl, const cd* right, long sr, const cd* A, long lda,
                              long sA, cd* C, long ldc, long sC, int inv_right) {
  const long bz = blockIdx.z;
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  const int c = blockIdx.y;
  if (r >= m) return;
  cd v = A[bz * sA + r + (long)c * lda];
  if (left) v = cmul(left[bz * sl + r], v);
  if (right) {
    cd f = right[bz * sr + c];
    v = inv_right ? cdiv(v, f) : cmul(v, f);
  }
  C[bz * sC + r + (long)c * ldc] = v;
}

void zdscale(hipStream_t s, int m, int n, const cd* left, long sl, const cd* right, long sr, int inv_right,
             const cd* A, long lda, long sA, cd* C, long ldc, long sC, int batch) {
  if (m <= 0 || n <= 0 || batch <= 0) return;
  dim3 grid(cdiv_up(m, 256), n, batch);
  dscale_kernel<<<grid, 256, 0, s>>>(m, n, left, sl, right, sr, A, lda, sA, C, ldc, sC, inv_right);
  launch_check("zdscale");
}

// Max |a_ij| (true modulus) per batch entry -> out[b] (double). One block per entry.
__global__ void maxabs_kernel(int m, int n, const cd* A, long lda, long sA, double* out) {
  const long bz = blockIdx.x;
  __shared__ double red[256];
  double mx = 0.0;
  const long total = (long)m * n;
  for (long e = threadIdx.x; e < total; e += blockDim.x) {
    int r = (int)(e % m), c = (int)(e / m);
    double v = cabsv(A[bz * sA + r + (long)c * lda]);
    mx = (v > mx || v != v) ? v : mx;
  }
  red[threadIdx.x] = mx;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      double o = red[threadIdx.x + w];
      double c = red[threadIdx.x];
      red[threadIdx.x] = (o > c || o != o) ? o : c;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[bz] = red[0];
}

void zmaxabs(hipStream_t s, int m, int n, const cd* A, long lda, long sA, double* out, int batch) {
  if (batch <= 0) return;
  maxabs_kernel<<<batch, 256, 0, s>>>(m, n, A, lda, sA, out);
  launch_check("zmaxabs");
}

}  // namespace vrc
