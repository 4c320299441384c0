// Batched complex128 non-Hermitian eigensolver for gfx950 (replaces the reference's
// LAPACKE_zgeev / magma_zgeev call, src/rcwa/MKLEigenSolver.hpp:45-55,
// src/gpu/RedhefferIntegratorGPU.cpp:216-229).
//
// Pipeline for a strided batch of n x n matrices:
//  1. Hessenberg reduction H = Q^H A Q: blocked Householder, panel of HB columns
//     reduced by one workgroup per matrix (the trailing-matrix product A*v is the
//     only memory-bound part), trailing update as three MFMA ZGEMMs.
//  2. Q formed explicitly from the stored reflectors (backward, blocked, ZGEMM).
//  3. Schur form T = Z^H H Z by a multishift QR sweep with tightly packed 3x3 bulges:
//     one workgroup per matrix; the bulge chain is chased inside a <=64x64 diagonal
//     window held in LDS, the window transform U is accumulated in LDS and applied
//     to the off-window rows/columns of H and to Z with in-kernel MFMA products.
//     Shifts are eigenvalues of the trailing block; blocks of size <= QR_NMIN are
//     finished by single-shift QR inside LDS.
//  4. Eigenvectors of T by a tiled back-substitution (64x64 tiles; one workgroup per
//     block column), then VR = Z * X (ZGEMM) and LAPACK zgeev normalisation.
#include <atomic>

#include "vrc_common.hpp"
#include "vrc_internal.hpp"
#include "vrc_context.hpp"
#include "vrc_ops.hpp"

namespace vrc {

constexpr double ULP = 2.220446049250313e-16;      // 2^-52
constexpr double SAFMIN = 2.2250738585072014e-308;
constexpr int HB = 64;         // Hessenberg panel width
constexpr int PT = 1024;       // threads of the Hessenberg panel workgroup (16 waves)
constexpr int GV_MAXG = 8;     // most column groups of the panel's matrix-vector product
constexpr int QT = 512;        // threads of the QR workgroup (8 waves; the window MFMAs use 4)
constexpr int QW = 64;         // maximal QR window
constexpr int NBUL = 16;       // most bulges per sweep (2 shifts each)
constexpr int QR_NMIN = 48;    // active blocks this small are finished in LDS
constexpr int EXC_SWEEPS = 6;  // sweeps without deflation before exceptional shifts
constexpr int AED_NIBBLE = 14; // skip the sweep when the window deflated more than this percentage

__device__ inline double wsum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Householder reflector G = I - tau v v^H, v = (1, x*scale), with G^H (alpha; x) = (beta; 0).
__device__ inline void house(cd alpha, double xnorm, double& beta, cd& tau, cd& scale) {
  if (xnorm == 0.0 && alpha.y == 0.0) {
    beta = alpha.x;
    tau = mk(0.0, 0.0);
    scale = mk(0.0, 0.0);
    return;
  }
  double nrm = hypot(hypot(alpha.x, alpha.y), xnorm);
  beta = alpha.x >= 0.0 ? -nrm : nrm;
  tau = mk((beta - alpha.x) / beta, -alpha.y / beta);
  scale = crecip(mk(alpha.x - beta, alpha.y));
}

// 1/sqrt(v) and 1/v for normal positive (nonzero) v: the hardware estimate (about 23 good
// bits) and one third-order Newton step, within about one unit in the last place.
__device__ __forceinline__ double rsqrt_nr(double v) {
  const double y = __builtin_amdgcn_rsq(v);
  const double e = fma(-v * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double rcp_nr(double v) {
  const double y = __builtin_amdgcn_rcp(v);
  const double e = fma(-v, y, 1.0);
  return fma(y, fma(e, e, e), y);
}
// Squares of values whose sum lies in this range neither overflow nor lose small parts.
__device__ __forceinline__ bool squares_safe(double s) { return s <= 0x1p800 && s >= 0x1p-800; }
__device__ __forceinline__ double wmax(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}
// |x / m|^2 for m > 0, the largest |re|, |im| of the values summed: their norm is m sqrt(sum) where
// the squares themselves are out of range (a norm that underflows to zero beside a reflector's
// nonzero first entry gives a reflector that is not unitary).
__device__ __forceinline__ double scaled_norm2(cd x, double m) { return cnorm2(mk(x.x / m, x.y / m)); }

// |x|_2 of x[0 .. n) where the squares are out of range; every wave computes it by itself.
__device__ inline double wave_norm(const cd* x, int n) {
  const int lane = threadIdx.x & 63;
  double m = 0.0, s = 0.0;
#pragma unroll 1
  for (int r = lane; r < n; r += 64) m = fmax(m, fmax(fabs(x[r].x), fabs(x[r].y)));
  m = wmax(m);
  if (!(m > 0.0)) m = 1.0;
#pragma unroll 1
  for (int r = lane; r < n; r += 64) s += scaled_norm2(x[r], m);
  return m * sqrt(wsum(s));
}

// The reflector of house() for |x|^2 = xn2 without a division or a square root in the
// chain: 1/|(alpha, x)| from one reciprocal square root, 1/(alpha - beta) as conj(d) / |d|^2.
// Out of range of the squares: house().
__device__ __forceinline__ void house_fast(cd alpha, double xn2, double& beta, cd& tau, cd& scale) {
  const double d2 = cnorm2(alpha) + xn2;
  if (__builtin_expect(!squares_safe(d2), 0)) {
    house(alpha, sqrt(xn2), beta, tau, scale);
    return;
  }
  const double rs = rsqrt_nr(d2);
  beta = -copysign(d2 * rs, alpha.x);
  const double rb = -copysign(rs, alpha.x);
  const double dx = alpha.x - beta, dy = alpha.y;
  const double id = rcp_nr(dx * dx + dy * dy);
  tau = mk((beta - alpha.x) * rb, -dy * rb);
  scale = mk(dx * id, -dy * id);
  if (xn2 == 0.0 && dy == 0.0) {
    beta = alpha.x;
    tau = scale = mk(0.0, 0.0);
  }
}

// The same for a vector spread over the wavefront (x: this lane's component).
__device__ __forceinline__ void wave_house(cd alpha, cd x, double& beta, cd& tau, cd& scale) {
  const double xn2 = wsum(cnorm2(x));
  if (__builtin_expect(squares_safe(cnorm2(alpha) + xn2), 1)) {
    house_fast(alpha, xn2, beta, tau, scale);
    return;
  }
  const double m = wmax(fmax(fabs(x.x), fabs(x.y)));
  house(alpha, m > 0.0 ? m * sqrt(wsum(scaled_norm2(x, m))) : sqrt(xn2), beta, tau, scale);
}

// The same for x = (y, z) (z = 0 for a 2-vector).
__device__ __forceinline__ void house_small(cd alpha, cd y, cd z, double& beta, cd& tau, cd& scale) {
  const double xn2 = cnorm2(y) + cnorm2(z);
  if (__builtin_expect(squares_safe(cnorm2(alpha) + xn2), 1))
    house_fast(alpha, xn2, beta, tau, scale);
  else
    house(alpha, hypot(cabsv(y), cabsv(z)), beta, tau, scale);
}

// ===================================================================== Hessenberg
constexpr int GV_W = 8;  // trailing-product loads in flight per thread

// One complex value read with the non-temporal hint (streamed once per column, not reused
// from cache).
typedef double vrc_d2 __attribute__((ext_vector_type(2)));
__device__ inline cd load_stream(const cd* p) {
  const vrc_d2 v = __builtin_nontemporal_load(reinterpret_cast<const vrc_d2*>(p));
  return mk(v.x, v.y);
}

// Sums v[0 .. NV) over the wavefront: the sum of v[k] ends in v[0] of the lanes with
// lane / (64 / NV) = k. Each step pairs the same lanes as a butterfly over all values would
// (the same sums), but lane halves keep half of the values each: 17 exchanges for 16 values
// instead of 96.
template <int NV>
__device__ __forceinline__ void wave_sums(double (&v)[NV]) {
  const int lane = threadIdx.x & 63;
  int off = 32;
#pragma unroll
  for (int h = NV / 2; h >= 1; h /= 2, off /= 2) {
    const bool up = lane & off;
#pragma unroll
    for (int k = 0; k < h; ++k) {
      const double keep = up ? v[h + k] : v[k], send = up ? v[k] : v[h + k];
      v[k] = keep + __shfl_xor(send, off, 64);
    }
  }
#pragma unroll
  for (; off >= 1; off /= 2) v[0] += __shfl_xor(v[0], off, 64);
}

// out[i] = sum_{r >= r0} conj(Vf[r, p+i]) x[r] for i < j (x in LDS): wave w reduces the
// columns i = w, w + PTT/64, ... (rows summed in increasing order within a lane). WIDE: NC = 8
// columns at a time share the waits for loads and lane exchanges. Otherwise one at a time, four
// loads in flight: the registers of the wide form would cost workgroups per CU (n = 882, 250
// matrices, four columns at a time: 263 -> 289 ms).
template <int PTT, bool WIDE>
__device__ void panel_multi_dot(int N, int r0, int p, int j, const cd* Vf, const cd* x, cd* out) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (WIDE) {
    constexpr int NW = PTT / 64, NC = 8, LPV = 32 / NC;  // LPV lanes share a sum
#pragma unroll 1
    for (int i0 = wave; i0 < j; i0 += NC * NW) {
      double s[2 * NC];
#pragma unroll
      for (int c = 0; c < 2 * NC; ++c) s[c] = 0.0;
#pragma unroll 1
      for (int r = r0 + lane; r < N; r += 64) {
        cd a[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const int i = i0 + c * NW;
          a[c] = Vf[r + (long)(p + (i < j ? i : i0)) * N];
        }
        const cd xb = x[r];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          s[2 * c] += a[c].x * xb.x + a[c].y * xb.y;
          s[2 * c + 1] += a[c].x * xb.y - a[c].y * xb.x;
        }
      }
      wave_sums<2 * NC>(s);
      const int k = lane / LPV, i = i0 + (k >> 1) * NW;
      if (lane % LPV == 0 && i < j) reinterpret_cast<double*>(out + i)[k & 1] = s[0];
    }
    __syncthreads();
    return;
  }
  for (int i = wave; i < j; i += PTT / 64) {
    const cd* vc = Vf + (long)(p + i) * N;
    double sr = 0.0, si = 0.0;
    int r = r0 + lane;
    for (; r + 192 < N; r += 256) {
      cd a[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) a[u] = vc[r + 64 * u];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const cd xb = x[r + 64 * u];
        sr += a[u].x * xb.x + a[u].y * xb.y;
        si += a[u].x * xb.y - a[u].y * xb.x;
      }
    }
    for (; r < N; r += 64) {
      const cd a = vc[r], xb = x[r];
      sr += a.x * xb.x + a.y * xb.y;
      si += a.x * xb.y - a.y * xb.x;
    }
    sr = wsum(sr);
    si = wsum(si);
    if (lane == 0) out[i] = mk(sr, si);
  }
  __syncthreads();
}

// acc - sum_{i < j} M[r + i ld] v[i], summed in increasing i with W loads in flight (the last
// group too: its loads stay within the j columns).
template <int W>
__device__ __forceinline__ cd sub_row_dot(cd acc, const cd* M, long ld, int r, int j, const cd* v) {
#pragma unroll 1
  for (int i = 0; i < j; i += W) {
    cd m[W], x[W];
#pragma unroll
    for (int u = 0; u < W; ++u) {
      const int c = i + u < j ? i + u : j - 1;
      m[u] = M[r + (long)c * ld];
      x[u] = v[c];
    }
#pragma unroll
    for (int u = 0; u < W; ++u) {
      const cd y = csub(acc, cmul(m[u], x[u]));
      acc.x = i + u < j ? y.x : acc.x;
      acc.y = i + u < j ? y.y : acc.y;
    }
  }
  return acc;
}

// Up to two matrices per CU; with more the narrow form runs four (N = 98, 640 matrices: wide 4.96,
// narrow 4.48 ms; N = 162: 11.9 and 11.0).
constexpr int GEHRD_WIDE_BATCH = 512;

// PTT threads: 1024 (16 waves) in general, 256 or 512 when N - 1 fits, so that several
// matrices share a CU (at most 128 VGPRs; the panel's T factor packed upper-triangular).
// WIDE (256 threads, up to two matrices per CU): a column is a chain of products that each wait
// for memory, so more of it is in flight in 256 VGPRs: 16 loads per row product, two column
// groups of the trailing product, eight columns per dot product. Same sums in the same order.
// Reduction of one batch, N = 98: 300 matrices 3.44 -> 3.00 ms; N = 162: 60 matrices
// 5.27 -> 4.34; N = 242: 100 matrices 11.0 -> 8.6, 200 matrices 12.8 -> 10.2.
template <int PTT, bool WIDE>
__global__ __launch_bounds__(PTT) __attribute__((amdgpu_waves_per_eu(WIDE ? 2 : 4))) void gehrd_panel_kernel(
    int N, int p, int nb, cd* A, long lda, long sA, cd* Vf, long sV, cd* Y, long sY, cd* Tp, long sT, cd* tau,
    long sTau) {
  const long b = blockIdx.x;
  A += b * sA;
  Vf += b * sV;
  Y += b * sY;
  Tp += b * sT;
  tau += b * sTau;
  extern __shared__ cd dyn[];
  cd* bvec = dyn;
  cd* vvec = dyn + N;
  __shared__ cd Tl[HB * (HB + 1) / 2];  // T(i, j), i <= j, at j (j + 1) / 2 + i
  __shared__ cd vec1[HB], vec2[HB];
  __shared__ double rn[PTT / 64];
  __shared__ cd gpart[PTT];  // per-thread partial sums of the column-split product
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  // rows below the panel; when they fit in the workgroup, the columns of the trailing
  // product are split over G groups of R threads (partial sums reduced through LDS)
  constexpr int SRD = WIDE ? 16 : 8;
  const int R = N - p - 1;
  const int G = (R > 0 && R <= PTT) ? (PTT / R < GV_MAXG ? PTT / R : GV_MAXG) : 1;

  for (int j = 0; j < nb; ++j) {
    const int c = p + j;
    if (t < j) vec1[t] = cconj(Vf[c + (long)(p + t) * N]);
    __syncthreads();
    // column c of A0*Q_j, rows below p (rows <= p are updated after the panel)
    for (int r = p + 1 + t; r < N; r += PTT) bvec[r] = sub_row_dot<SRD>(A[r + (long)c * lda], Y, N, r, j, vec1);
    __syncthreads();
    if (j > 0) {
      // left transform by Q_j^H on rows >= p+1
      panel_multi_dot<PTT, WIDE>(N, p + 1, p, j, Vf, bvec, vec2);
      if (t < j) {
        cd s = mk(0.0, 0.0);
#pragma unroll 1
        for (int l0 = 0; l0 <= t; l0 += 4) {
          cd T4[4], z4[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int l = l0 + u <= t ? l0 + u : t;
            T4[u] = Tl[t * (t + 1) / 2 + l];
            z4[u] = vec2[l];
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const cd y = cadd(s, cmul(cconj(T4[u]), z4[u]));
            s.x = l0 + u <= t ? y.x : s.x;
            s.y = l0 + u <= t ? y.y : s.y;
          }
        }
        vec1[t] = s;
      }
      __syncthreads();
      for (int r = p + 1 + t; r < N; r += PTT) bvec[r] = sub_row_dot<SRD>(bvec[r], Vf + (long)p * N, N, r, j, vec1);
      __syncthreads();
    }
    // final entries of column c and the reflector from rows c+1..N-1
    double part = 0.0;
    for (int r = p + 1 + t; r < N; r += PTT) {
      if (r <= c) A[r + (long)c * lda] = bvec[r];
      if (r >= c + 2) part += cnorm2(bvec[r]);
    }
    part = wsum(part);
    if (lane == 0) rn[wave] = part;
    __syncthreads();
    double xn2 = 0.0;
    for (int w = 0; w < PTT / 64; ++w) xn2 += rn[w];
    double xnorm = sqrt(xn2);
    // Not in the wide form: any use of xn2 there costs 24 registers and 3 to 8 % of the reduction
    // (N = 162, 2 matrices 3.31 -> 3.57 ms), so a column whose squares underflow beside a nonzero
    // entry is not reduced accurately for N <= 257 in launches of up to 512 matrices.
    if constexpr (!WIDE)
      if (__builtin_expect(!squares_safe(xn2), 0)) xnorm = wave_norm(bvec + c + 2, N - c - 2);
    double beta;
    cd tv, scale;
    house(bvec[c + 1], xnorm, beta, tv, scale);
    const bool ident = (tv.x == 0.0 && tv.y == 0.0);
    for (int r = t; r < N; r += PTT) {
      cd v;
      if (r <= c) v = mk(0.0, 0.0);
      else if (r == c + 1) v = mk(1.0, 0.0);
      else v = ident ? mk(0.0, 0.0) : cmul(bvec[r], scale);
      vvec[r] = v;
      Vf[r + (long)c * N] = v;
      if (r == c + 1) A[r + (long)c * lda] = ident ? bvec[r] : mk(beta, 0.0);
      else if (r > c + 1) A[r + (long)c * lda] = mk(0.0, 0.0);
    }
    if (t == 0) tau[c] = tv;
    __syncthreads();
    // z = V_j^H v  (rows >= c+1)
    if (j > 0) panel_multi_dot<PTT, WIDE>(N, c + 1, p, j, Vf, vvec, vec2);
    // y_j = tau*(A0[:, c+1:] v - Y_j z) for the rows below p (the rows above are one
    // ZGEMM after the panel). The trailing-matrix product is the memory-bound part.
    if (R > 0 && R <= PTT) {
      // thread (g, i): row p+1+i, columns c+1+GV_W g+GV_W Gk .. +GV_W (GV_W loads in flight)
      const int g = t / R, i = t - g * R;
      double sr = 0.0, si = 0.0;
      if (g < G) {
        const int r = p + 1 + i;
        constexpr int GB = WIDE ? 2 : 1;  // groups of GV_W columns in flight
#pragma unroll 1
        for (int col0 = c + 1 + GV_W * g; col0 < N; col0 += GB * GV_W * G) {
          cd a[GB * GV_W];
#pragma unroll
          for (int u = 0; u < GB * GV_W; ++u) {
            const int col = col0 + u % GV_W + (u / GV_W) * GV_W * G;
            a[u] = load_stream(A + r + (long)(col < N ? col : N - 1) * lda);
          }
#pragma unroll
          for (int u = 0; u < GB * GV_W; ++u) {
            const int col = col0 + u % GV_W + (u / GV_W) * GV_W * G;
            const bool in = col < N;
            const cd v = vvec[in ? col : N - 1];
            const double dr = a[u].x * v.x - a[u].y * v.y, di = a[u].x * v.y + a[u].y * v.x;
            sr = in ? sr + dr : sr;
            si = in ? si + di : si;
          }
        }
      }
      gpart[t] = mk(sr, si);
      __syncthreads();
      if (t < R) {
        const int r = p + 1 + t;
        cd acc = gpart[t];
        for (int q = 1; q < G; ++q) acc = cadd(acc, gpart[q * R + t]);
        acc = sub_row_dot<SRD>(acc, Y, N, r, j, vec2);
        Y[r + (long)j * N] = cmul(tv, acc);
      }
    } else
    for (int rb = p + 1 + t; rb < N; rb += 4 * PTT) {
      double gr[4] = {0.0, 0.0, 0.0, 0.0}, gi[4] = {0.0, 0.0, 0.0, 0.0};
      int col = c + 1;
      for (; col + 3 < N; col += 4) {
        cd v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = vvec[col + u];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = rb + PTT * q;
          if (r < N) {
            const cd* ar = A + r + (long)col * lda;
            cd a[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) a[u] = ar[(long)u * lda];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              gr[q] += a[u].x * v[u].x - a[u].y * v[u].y;
              gi[q] += a[u].x * v[u].y + a[u].y * v[u].x;
            }
          }
        }
      }
      for (; col < N; ++col) {
        const cd v = vvec[col];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = rb + PTT * q;
          if (r < N) {
            const cd a = A[r + (long)col * lda];
            gr[q] += a.x * v.x - a.y * v.y;
            gi[q] += a.x * v.y + a.y * v.x;
          }
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = rb + PTT * q;
        if (r < N) {
          cd acc = mk(gr[q], gi[q]);
          for (int i = 0; i < j; ++i) acc = csub(acc, cmul(Y[r + (long)i * N], vec2[i]));
          Y[r + (long)j * N] = cmul(tv, acc);
        }
      }
    }
    if (t < j) {
      cd s = mk(0.0, 0.0);
#pragma unroll 1
      for (int l0 = t; l0 < j; l0 += 4) {
        cd T4[4], z4[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int l = l0 + u < j ? l0 + u : j - 1;
          T4[u] = Tl[l * (l + 1) / 2 + t];
          z4[u] = vec2[l];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const cd y = cadd(s, cmul(T4[u], z4[u]));
          s.x = l0 + u < j ? y.x : s.x;
          s.y = l0 + u < j ? y.y : s.y;
        }
      }
      Tl[j * (j + 1) / 2 + t] = cneg(cmul(tv, s));
    }
    if (t == 0) Tl[j * (j + 1) / 2 + j] = tv;
    __syncthreads();
  }
  for (int e = t; e < nb * nb; e += PTT) {
    int i = e % nb, jj = e / nb;
    Tp[i + (long)jj * HB] = (i <= jj) ? Tl[jj * (jj + 1) / 2 + i] : mk(0.0, 0.0);
  }
}

// ---- the same panel spread over many workgroups, three launches per column
// With few matrices the one-workgroup panel reads each trailing matrix through one CU (about
// 100 GB/s) once per column. Here every step of a column runs over blocks of GS_R rows, and
// the trailing product over tiles of GS_G rows and GS_C columns, so that the chip's bandwidth
// is used; a step ends where the next needs a sum over all rows (one launch each, no waits
// between workgroups). Per matrix, work holds the vector b, the row blocks' partial sums and
// the column tiles' partial products.
constexpr int GS_R = 64, GS_G = 256, GS_C = 64;
struct GehrdWork {  // offsets (in cd) into a matrix's work area
  int nblk, nsp;    // row blocks and column tiles at the panel's first column
  long dots, z, norm, part, size;
  __host__ __device__ GehrdWork(int N, int p)
      : nblk((N - p - 1 + GS_R - 1) / GS_R), nsp((N - p - 1 + GS_C - 1) / GS_C) {
    dots = N;
    z = dots + (long)nblk * HB;
    norm = z + (long)nblk * HB;
    part = norm + nblk;
    size = part + (long)nsp * N;
  }
};

// out[i] = sum over the blocks of src[blk * HB + i], i < n (256 threads; ends with a barrier).
__device__ inline void sum_blocks(const cd* src, int nblk, int n, cd (*red)[64], cd* out) {
  const int i = threadIdx.x & 63, q = threadIdx.x >> 6;
  cd acc = mk(0.0, 0.0);
  if (i < n)
    for (int k = q; k < nblk; k += 4) acc = cadd(acc, src[(long)k * HB + i]);
  red[q][i] = acc;
  __syncthreads();
  if (q == 0) out[i] = cadd(cadd(red[0][i], red[1][i]), cadd(red[2][i], red[3][i]));
  __syncthreads();
}

// dst[i] = sum over the block's rows of conj(V[r, p + i]) x(r), i < j; the wave's lanes hold rows.
__device__ inline void block_dots(int N, int p, int j, const cd* V, int r, cd x, cd* dst) {
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  for (int i0 = q; i0 < j; i0 += 16) {
    cd v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      v[u] = (r < N && i0 + 4 * u < j) ? V[r + (long)(p + i0 + 4 * u) * N] : mk(0.0, 0.0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const cd d = cmulc(x, v[u]);
      const double sr = wsum(d.x), si = wsum(d.y);
      if (lane == 0 && i0 + 4 * u < j) dst[i0 + 4 * u] = mk(sr, si);
    }
  }
}

// Column j's first step: y and T of column j - 1 completed, b = column c of A0 Q_j (rows below
// p), and the blocks' parts of V^H b. j == nb: only the completion.
__global__ __launch_bounds__(256) void gehrd_col_a_kernel(int N, int p, int nb, int j, const cd* A, long lda, long sA,
                                                          const cd* V, long sV, cd* Y, long sY, cd* Tp, long sT,
                                                          const cd* tau, long sTau, cd* work, GehrdWork gw) {
  const long m = blockIdx.y;
  A += m * sA;
  V += m * sV;
  Y += m * sY;
  Tp += m * sT;
  tau += m * sTau;
  work += m * gw.size;
  __shared__ cd red[4][64], zs[64], vc[64], bs[64], ys[64];
  const int t = threadIdx.x, tr = t & 63, q = t >> 6;
  const int blk = blockIdx.x, c = p + j;
  const int r = p + 1 + blk * GS_R + tr;
  const int jm = j > 0 ? j - 1 : 0;
  if (t < 64) vc[t] = (t < j && j < nb) ? cconj(V[c + (long)(p + t) * N]) : mk(0.0, 0.0);
  sum_blocks(work + gw.z, gw.nblk, jm, red, zs);
  cd ay = mk(0.0, 0.0), ab = mk(0.0, 0.0);
  if (r < N) {
    if (j > 0) {
      const int sp = (N - (c - 1) - 1 + GS_C - 1) / GS_C;
      for (int k = q; k < sp; k += 4) ay = cadd(ay, work[gw.part + (long)k * N + r]);
    }
    for (int i = q; i < jm; i += 4) {
      const cd y = Y[r + (long)i * N];
      ay = csub(ay, cmul(y, zs[i]));
      ab = cadd(ab, cmul(y, vc[i]));
    }
  }
  red[q][tr] = ay;
  __syncthreads();
  if (q == 0 && j > 0) {
    const cd y = cmul(tau[c - 1], cadd(cadd(red[0][tr], red[1][tr]), cadd(red[2][tr], red[3][tr])));
    ys[tr] = y;
    if (r < N) Y[r + (long)jm * N] = y;
  }
  __syncthreads();
  red[q][tr] = ab;
  __syncthreads();
  if (blk == 0 && j > 0) {  // T(0 .. j-1, j-1)
    const cd tv = tau[c - 1];
    if (t < HB) {
      cd s = mk(0.0, 0.0);
      for (int l = t; l < jm; ++l) s = cadd(s, cmul(Tp[t + (long)l * HB], zs[l]));
      Tp[t + (long)jm * HB] = t < jm ? cneg(cmul(tv, s)) : (t == jm ? tv : mk(0.0, 0.0));
    }
  }
  if (j >= nb) return;
  if (q == 0) {
    cd b = mk(0.0, 0.0);
    if (r < N) {
      b = csub(A[r + (long)c * lda], cadd(cadd(red[0][tr], red[1][tr]), cadd(red[2][tr], red[3][tr])));
      if (j > 0) b = csub(b, cmul(ys[tr], vc[jm]));
      work[r] = b;
    }
    bs[tr] = b;
  }
  __syncthreads();
  block_dots(N, p, j, V, r, bs[tr], work + gw.dots + (long)blk * HB);
}

// Second step: b -= V T^H (V^H b), the finished entries of column c (rows up to c), and the
// blocks' parts of the norm of the rest.
__global__ __launch_bounds__(256) void gehrd_col_b_kernel(int N, int p, int j, cd* A, long lda, long sA, const cd* V,
                                                          long sV, const cd* Tp, long sT, cd* work, GehrdWork gw) {
  const long m = blockIdx.y;
  A += m * sA;
  V += m * sV;
  Tp += m * sT;
  work += m * gw.size;
  __shared__ cd red[4][64], ds[64], ss[64];
  const int t = threadIdx.x, tr = t & 63, q = t >> 6;
  const int blk = blockIdx.x, c = p + j;
  const int r = p + 1 + blk * GS_R + tr;
  cd ab = mk(0.0, 0.0);
  if (j > 0) {
    sum_blocks(work + gw.dots, gw.nblk, j, red, ds);
    cd s = mk(0.0, 0.0);
    if (tr < j)
      for (int l = q; l <= tr; l += 4) s = cadd(s, cmulc(ds[l], Tp[l + (long)tr * HB]));
    red[q][tr] = s;
    __syncthreads();
    if (q == 0) ss[tr] = cadd(cadd(red[0][tr], red[1][tr]), cadd(red[2][tr], red[3][tr]));
    __syncthreads();
    if (r < N)
      for (int i = q; i < j; i += 4) ab = cadd(ab, cmul(V[r + (long)(p + i) * N], ss[i]));
  }
  red[q][tr] = ab;
  __syncthreads();
  if (q > 0) return;
  cd x = mk(0.0, 0.0);
  if (r < N) {
    cd b = work[r];
    if (j > 0) {
      b = csub(b, cadd(cadd(red[0][tr], red[1][tr]), cadd(red[2][tr], red[3][tr])));
      work[r] = b;
    }
    if (r <= c) A[r + (long)c * lda] = b;
    if (r >= c + 2) x = b;
  }
  // the block's part: a sum of squares and the scale of the values squared (0: all zero)
  double nn = wsum(cnorm2(x)), big = 1.0;
  if (!squares_safe(nn)) {
    big = wmax(fmax(fabs(x.x), fabs(x.y)));
    if (big > 0.0) nn = wsum(scaled_norm2(x, big));
  }
  if (tr == 0) work[gw.norm + blk] = mk(nn, big);
}

// Third step: the reflector (every workgroup computes it), the trailing product's tiles
// (workgroups below ngemv: rows x columns), and by the rest its vector in V, column c of A and
// the blocks' parts of V^H v.
__global__ __launch_bounds__(256) void gehrd_col_c_kernel(int N, int p, int j, cd* A, long lda, long sA, cd* V, long sV,
                                                          cd* tau, long sTau, cd* work, GehrdWork gw, int nrow,
                                                          int ngemv) {
  const long m = blockIdx.y;
  A += m * sA;
  V += m * sV;
  tau += m * sTau;
  work += m * gw.size;
  __shared__ cd vs[GS_C];
  const int t = threadIdx.x, lane = t & 63, q = t >> 6;
  const int c = p + j;
  double nn = 0.0, big = 0.0;
  for (int k = lane; k < gw.nblk; k += 64) big = fmax(big, work[gw.norm + k].y);
  big = wmax(big);
  for (int k = lane; k < gw.nblk; k += 64) {
    const cd part = work[gw.norm + k];
    const double f = big > 0.0 ? part.y / big : 1.0;
    nn += part.x * (f * f);
  }
  const double xnorm = (big > 0.0 ? big : 1.0) * sqrt(wsum(nn));
  const cd alpha = work[c + 1];
  double beta;
  cd tv, scale;
  house(alpha, xnorm, beta, tv, scale);
  const bool ident = tv.x == 0.0 && tv.y == 0.0;
  auto vec = [&](int r) {
    if (r <= c || r >= N) return mk(0.0, 0.0);
    if (r == c + 1) return mk(1.0, 0.0);
    return ident ? mk(0.0, 0.0) : cmul(work[r], scale);
  };
  if ((int)blockIdx.x < ngemv) {
    const int rt = blockIdx.x % nrow, sp = blockIdx.x / nrow;
    const int c0 = c + 1 + sp * GS_C;
    if (t < GS_C) vs[t] = vec(c0 + t);
    __syncthreads();
    const int r = p + 1 + rt * GS_G + t;
    if (r >= N) return;
    const int nc = N - c0 < GS_C ? N - c0 : GS_C;
    const cd* ar = A + r + (long)c0 * lda;
    double sr = 0.0, si = 0.0;
    int k = 0;
    for (; k + 8 <= nc; k += 8) {
      cd a[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] = ar[(long)(k + u) * lda];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const cd v = vs[k + u];
        sr += a[u].x * v.x - a[u].y * v.y;
        si += a[u].x * v.y + a[u].y * v.x;
      }
    }
    for (; k < nc; ++k) {
      const cd a = ar[(long)k * lda], v = vs[k];
      sr += a.x * v.x - a.y * v.y;
      si += a.x * v.y + a.y * v.x;
    }
    work[gw.part + (long)sp * N + r] = mk(sr, si);
    return;
  }
  const int blk = blockIdx.x - ngemv;
  const int r = p + 1 + blk * GS_R + lane;
  const cd v = vec(r);
  if (q == 0 && r < N) {
    V[r + (long)c * N] = v;
    if (r == c + 1)
      A[r + (long)c * lda] = ident ? alpha : mk(beta, 0.0);
    else if (r > c + 1)
      A[r + (long)c * lda] = mk(0.0, 0.0);
  }
  if (blk == 0 && t == 0) tau[c] = tv;
  block_dots(N, p, j, V, r, v, work + gw.z + (long)blk * HB);
}

// Spread the panel when the matrices alone would leave most CUs idle and are too large for the
// wide form of the panel in one workgroup. Hessenberg stage, ms, one workgroup / spread:
// N = 242 (wide) 1 matrix 6.0 / 6.2, 10 6.6 / 6.7, 40 7.9 / 8.8, 60 8.1 / 9.8; N = 258 8 7.7 / 7.1,
// 24 8.2 / 8.2, 64 9.1 / 10.4; N = 338 24 13.0 / 11.4, 40 13.8 / 13.0, 56 14.4 / 14.5, 64 14.5 / 15.1;
// N = 450 8 20.5 / 13.8, 64 26.4 / 24.6, 80 27.6 / 28.1; N = 882 8 103 / 35, 64 129 / 104, 96 147 / 144,
// 112 156 / 164. The line follows the crossings up to N = 373 and stays at 64 matrices from there.
static bool gehrd_spread(int n, int batch) { return n > 257 && batch <= 64 && 20 * batch <= 7 * (n - 190); }

static int n_reflectors(int n) { return n >= 3 ? n - 2 : 0; }

// A <- H (Hessenberg, zeros below the subdiagonal). Vf (n x n) receives the
// reflector vectors by column, Tall (npanel x HB x HB) the panel T factors.
static void gehrd(hipStream_t s, int n, cd* A, long lda, long sA, cd* Vf, cd* Tall, int batch, Workspace& ws) {
  const int nref = n_reflectors(n);
  if (nref == 0) return;
  const int npanel = cdiv_up(nref, HB);
  DevBuf Yb = ws.get(sizeof(cd) * (size_t)n * HB * batch);
  DevBuf taub = ws.get(sizeof(cd) * (size_t)n * batch);
  DevBuf Wb = ws.get(sizeof(cd) * (size_t)HB * n * batch);
  DevBuf W2b = ws.get(sizeof(cd) * (size_t)HB * n * batch);
  cd* Y = Yb.as<cd>();
  cd* W = Wb.as<cd>();
  cd* W2 = W2b.as<cd>();
  const long sV = (long)n * n, sY = (long)n * HB, sT = (long)npanel * HB * HB, sW = (long)HB * n;
  const cd one = mk(1.0, 0.0), mone = mk(-1.0, 0.0), zero = mk(0.0, 0.0);
  const bool spread = gehrd_spread(n, batch);
  DevBuf workb;
  if (spread) workb = ws.get(sizeof(cd) * (size_t)GehrdWork(n, 0).size * batch);
  for (int p = 0; p < nref; p += HB) {
    const int nb = nref - p < HB ? nref - p : HB;
    cd* Tp = Tall + (long)(p / HB) * HB * HB;
    if (spread) {
      const GehrdWork gw(n, p);
      cd* work = workb.as<cd>();
      const int nrow = cdiv_up(n - p - 1, GS_G);
      const dim3 rows(gw.nblk, batch);
      for (int j = 0; j <= nb; ++j) {
        gehrd_col_a_kernel<<<rows, 256, 0, s>>>(n, p, nb, j, A, lda, sA, Vf, sV, Y, sY, Tp, sT, taub.as<cd>(), n, work,
                                                gw);
        if (j == nb) break;
        gehrd_col_b_kernel<<<rows, 256, 0, s>>>(n, p, j, A, lda, sA, Vf, sV, Tp, sT, work, gw);
        const int ngemv = nrow * cdiv_up(n - (p + j) - 1, GS_C);
        gehrd_col_c_kernel<<<dim3(ngemv + gw.nblk, batch), 256, 0, s>>>(n, p, j, A, lda, sA, Vf, sV, taub.as<cd>(), n,
                                                                        work, gw, nrow, ngemv);
      }
    } else if (n - 1 <= 256 && batch <= GEHRD_WIDE_BATCH)
      gehrd_panel_kernel<256, true><<<batch, 256, 2 * sizeof(cd) * n, s>>>(n, p, nb, A, lda, sA, Vf, sV, Y, sY, Tp,
                                                                           sT, taub.as<cd>(), n);
    else if (n - 1 <= 256)
      gehrd_panel_kernel<256, false><<<batch, 256, 2 * sizeof(cd) * n, s>>>(n, p, nb, A, lda, sA, Vf, sV, Y, sY, Tp,
                                                                            sT, taub.as<cd>(), n);
    else if (n - 1 <= 512)
      gehrd_panel_kernel<512, false><<<batch, 512, 2 * sizeof(cd) * n, s>>>(n, p, nb, A, lda, sA, Vf, sV, Y, sY, Tp,
                                                                            sT, taub.as<cd>(), n);
    else
      gehrd_panel_kernel<PT, false><<<batch, PT, 2 * sizeof(cd) * n, s>>>(n, p, nb, A, lda, sA, Vf, sV, Y, sY, Tp,
                                                                          sT, taub.as<cd>(), n);
    launch_check("gehrd_panel");
    // rows 0..p: Y = A0 V T, then the panel columns' A0 Q = A0 - Y V^H
    zgemm_strided(s, OP_N, OP_N, p + 1, nb, n - p - 1, one, A + (long)(p + 1) * lda, lda, sA,
                  Vf + (p + 1) + (long)p * n, n, sV, zero, W, n, sW, batch);
    zgemm_strided(s, OP_N, OP_N, p + 1, nb, nb, one, W, n, sW, Tp, HB, sT, zero, Y, n, sY, batch);
    if (nb > 1)
      zgemm_strided(s, OP_N, OP_C, p + 1, nb - 1, nb, mone, Y, n, sY, Vf + (p + 1) + (long)p * n, n, sV, one,
                    A + (long)(p + 1) * lda, lda, sA, batch);
    const int c0 = p + nb, ncols = n - c0;
    if (ncols <= 0) continue;
    zgemm_strided(s, OP_N, OP_C, n, ncols, nb, mone, Y, n, sY, Vf + c0 + (long)p * n, n, sV, one,
                  A + (long)c0 * lda, lda, sA, batch);
    zgemm_strided(s, OP_C, OP_N, nb, ncols, n - p - 1, one, Vf + (p + 1) + (long)p * n, n, sV,
                  A + (p + 1) + (long)c0 * lda, lda, sA, zero, W, HB, sW, batch);
    zgemm_strided(s, OP_C, OP_N, nb, ncols, nb, one, Tp, HB, sT, W, HB, sW, zero, W2, HB, sW, batch);
    zgemm_strided(s, OP_N, OP_N, n - p - 1, ncols, nb, mone, Vf + (p + 1) + (long)p * n, n, sV, W2, HB, sW, one,
                  A + (p + 1) + (long)c0 * lda, lda, sA, batch);
  }
}

// Q = H_0 H_1 ... H_{nref-1} into Z (n x n).
static void orghr(hipStream_t s, int n, const cd* Vf, const cd* Tall, cd* Z, long ldz, long sZ, int batch,
                  Workspace& ws) {
  zset(s, n, n, mk(1.0, 0.0), mk(0.0, 0.0), Z, ldz, sZ, batch);
  const int nref = n_reflectors(n);
  if (nref == 0) return;
  const int npanel = cdiv_up(nref, HB);
  DevBuf Wb = ws.get(sizeof(cd) * (size_t)HB * n * batch);
  DevBuf W2b = ws.get(sizeof(cd) * (size_t)HB * n * batch);
  const long sV = (long)n * n, sT = (long)npanel * HB * HB, sW = (long)HB * n;
  const cd one = mk(1.0, 0.0), mone = mk(-1.0, 0.0), zero = mk(0.0, 0.0);
  for (int pi = npanel - 1; pi >= 0; --pi) {
    const int p = pi * HB;
    const int nb = nref - p < HB ? nref - p : HB;
    const int m = n - p - 1;
    const cd* V = Vf + (p + 1) + (long)p * n;
    cd* Zs = Z + (p + 1) + (long)(p + 1) * ldz;
    zgemm_strided(s, OP_C, OP_N, nb, m, m, one, V, n, sV, Zs, ldz, sZ, zero, Wb.as<cd>(), HB, sW, batch);
    zgemm_strided(s, OP_N, OP_N, nb, m, nb, one, Tall + (long)pi * HB * HB, HB, sT, Wb.as<cd>(), HB, sW, zero,
                  W2b.as<cd>(), HB, sW, batch);
    zgemm_strided(s, OP_N, OP_N, m, m, nb, mone, V, n, sV, W2b.as<cd>(), HB, sW, one, Zs, ldz, sZ, batch);
  }
}

// ===================================================================== LDS matrix products
typedef cd LdsMat[QW][QW + 1];

// acc = op(A) * B over K = 4 * ks (<= 64) for the 64x64 output tile; CT selects
// op(A)(i,k) = conj(A[k][i]). Windows narrower than 64 (zero padded) take fewer k steps.
template <bool CT, bool FULL = true>
__device__ __forceinline__ void mm64(const LdsMat& As, const LdsMat& Bs, int ks, d4 (&accR)[2][2],
                                     d4 (&accI)[2][2]) {
  if (FULL) ks = QW / 4;  // compile-time trip count for the full window
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wr = wave >> 1, wc = wave & 1;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      accR[i][j] = d4{0.0, 0.0, 0.0, 0.0};
      accI[i][j] = d4{0.0, 0.0, 0.0, 0.0};
    }
  for (int s = 0; s < ks; ++s) {
    const int kr = 4 * s + (lane >> 4);
    double ar[2], ai[2], nai[2], br[2], bi[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int i = wr * 32 + q * 16 + (lane & 15);
      cd a = CT ? cconj(As[kr][i]) : As[i][kr];
      ar[q] = a.x;
      ai[q] = a.y;
      nai[q] = -a.y;
      const int j = wc * 32 + q * 16 + (lane & 15);
      cd bb = Bs[kr][j];
      br[q] = bb.x;
      bi[q] = bb.y;
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
}

// Calls f(i, j, value) for every output element owned by this thread.
template <class F>
__device__ __forceinline__ void mm64_for_each(const d4 (&accR)[2][2], const d4 (&accI)[2][2], F f) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wr = wave >> 1, wc = wave & 1;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int ii = wr * 32 + i * 16 + (lane >> 4) + 4 * r;
        const int jj = wc * 32 + j * 16 + (lane & 15);
        f(ii, jj, mk(accR[i][j][r], accI[i][j][r]));
      }
}

// The same product on eight waves (QR workgroup): wave w owns rows 32*(w>>2) .. +32 and
// columns 16*(w&3) .. +16 of the 64x64 output (two 16x16 blocks).
static_assert(QT == 512, "the QR window multiply and its staging assume eight waves");
template <bool CT, bool FULL>
__device__ __forceinline__ void mm64w8(const LdsMat& As, const LdsMat& Bs, int ks, d4 (&accR)[2], d4 (&accI)[2]) {
  if (FULL) ks = QW / 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wr = wave >> 2, wc = wave & 3;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    accR[i] = d4{0.0, 0.0, 0.0, 0.0};
    accI[i] = d4{0.0, 0.0, 0.0, 0.0};
  }
  for (int s = 0; s < ks; ++s) {
    const int kr = 4 * s + (lane >> 4);
    double ar[2], ai[2], nai[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int i = wr * 32 + q * 16 + (lane & 15);
      cd a = CT ? cconj(As[kr][i]) : As[i][kr];
      ar[q] = a.x;
      ai[q] = a.y;
      nai[q] = -a.y;
    }
    const cd bb = Bs[kr][wc * 16 + (lane & 15)];
    const double br = bb.x, bi = bb.y;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      accR[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], br, accR[i], 0, 0, 0);
      accR[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(nai[i], bi, accR[i], 0, 0, 0);
      accI[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], bi, accI[i], 0, 0, 0);
      accI[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[i], br, accI[i], 0, 0, 0);
    }
  }
}

template <class F>
__device__ __forceinline__ void mm64w8_for_each(const d4 (&accR)[2], const d4 (&accI)[2], F f) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wr = wave >> 2, wc = wave & 3;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ii = wr * 32 + i * 16 + (lane >> 4) + 4 * r;
      const int jj = wc * 16 + (lane & 15);
      f(ii, jj, mk(accR[i][r], accI[i][r]));
    }
}

// M[r0:r0+w, c0:c1] <- U^H * M[...]  (U: w x w in LDS, zero padded), chunk buffer C;
// QT threads. The next 64-column chunk is fetched into registers while the current one
// is multiplied.
__device__ void apply_left_u(const LdsMat& U, LdsMat& C, int w, cd* M, long ld, int r0, int c0, int c1) {
  const int t = threadIdx.x;
  const int k = t & 63, j0 = t >> 6;  // element (k, j0 + 8q) of a chunk, q < 8
  cd pre[8];
  if (c0 < c1) {
    const int cw = c1 - c0 < QW ? c1 - c0 : QW;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      pre[q] = (k < w && j0 + 8 * q < cw) ? M[(r0 + k) + (long)(c0 + j0 + 8 * q) * ld] : mk(0.0, 0.0);
  }
  for (int cc = c0; cc < c1; cc += QW) {
    const int cw = c1 - cc < QW ? c1 - cc : QW;
#pragma unroll
    for (int q = 0; q < 8; ++q) C[k][j0 + 8 * q] = pre[q];
    __syncthreads();
    const int cn = cc + QW;
    if (cn < c1) {
      const int cwn = c1 - cn < QW ? c1 - cn : QW;
#pragma unroll
      for (int q = 0; q < 8; ++q)
        pre[q] = (k < w && j0 + 8 * q < cwn) ? M[(r0 + k) + (long)(cn + j0 + 8 * q) * ld] : mk(0.0, 0.0);
    }
    d4 aR[2], aI[2];
    if (w == QW)
      mm64w8<true, true>(U, C, QW / 4, aR, aI);
    else
      mm64w8<true, false>(U, C, (w + 3) >> 2, aR, aI);
    mm64w8_for_each(aR, aI, [&](int i, int j, cd v) {
      if (i < w && j < cw) M[(r0 + i) + (long)(cc + j) * ld] = v;
    });
    __syncthreads();
  }
}
// M[r0:r1, c0:c0+w] <- M[...] * U, 64-row chunks, next chunk prefetched into registers.
__device__ void apply_right_u(const LdsMat& U, LdsMat& C, int w, cd* M, long ld, int r0, int r1, int c0) {
  const int t = threadIdx.x;
  const int i = t & 63, k0 = t >> 6;  // element (i, k0 + 8q) of a chunk, q < 8
  cd pre[8];
  if (r0 < r1) {
    const int rh = r1 - r0 < QW ? r1 - r0 : QW;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      pre[q] = (i < rh && k0 + 8 * q < w) ? M[(r0 + i) + (long)(c0 + k0 + 8 * q) * ld] : mk(0.0, 0.0);
  }
  for (int rr = r0; rr < r1; rr += QW) {
    const int rh = r1 - rr < QW ? r1 - rr : QW;
#pragma unroll
    for (int q = 0; q < 8; ++q) C[i][k0 + 8 * q] = pre[q];
    __syncthreads();
    const int rn = rr + QW;
    if (rn < r1) {
      const int rhn = r1 - rn < QW ? r1 - rn : QW;
#pragma unroll
      for (int q = 0; q < 8; ++q)
        pre[q] = (i < rhn && k0 + 8 * q < w) ? M[(rn + i) + (long)(c0 + k0 + 8 * q) * ld] : mk(0.0, 0.0);
    }
    d4 aR[2], aI[2];
    if (w == QW)
      mm64w8<false, true>(C, U, QW / 4, aR, aI);
    else
      mm64w8<false, false>(C, U, (w + 3) >> 2, aR, aI);
    mm64w8_for_each(aR, aI, [&](int ii, int j, cd v) {
      if (ii < rh && j < w) M[(rr + ii) + (long)(c0 + j) * ld] = v;
    });
    __syncthreads();
  }
}
// ===================================================================== QR iteration
// The QR workgroup's LDS: the W x W window, its accumulated transform U and the bulge
// and reduction scratch. W = 64 with T = 512 threads fills most of a CU's LDS (one
// workgroup per CU); W = 48 with T = 256 stays under half of it, so two workgroups (two
// matrices) share a CU and one's serial bulge chase overlaps the other's window products.
template <int W>
using QMat = cd[W][W + 1];
template <int W, int T>
struct QrLds {
  QMat<W> Hw;
  QMat<W> U;
  cd shifts[2 * NBUL];
  int redi[T];
  cd aedv[64];  // written by every lane of a wavefront
  int ctl[4];
};
static_assert(sizeof(QrLds<48, 256>) <= 80 * 1024, "two W = 48 QR workgroups must fit one CU's LDS");
static_assert(sizeof(QrLds<32, 128>) <= 40 * 1024, "four W = 32 QR workgroups must fit one CU's LDS");

// Window products from registers (no LDS chunk buffer, no barrier): with the 16x16x4 FP64
// MFMA, lane l supplies A[l & 15][l >> 4] and B[l >> 4][l & 15] and holds
// D[(l >> 4) + 4 q][l & 15], q < 4. Both products are formed transposed so that a lane's
// global loads and stores run along a column (16 consecutive rows per instruction).
//
// M[r0:r0+w, c0:c1] <- U^H M[...]: as D = M^T conj(U) per 16 columns; the wave takes the
// 16-column strips first, first + step, ..., reads their w rows into registers and writes
// them back.
template <int W>
__device__ void apply_left_reg(const QMat<W>& U, int w, cd* M, long ld, int r0, int c0, int c1, int first,
                               int step) {
  constexpr int KS = W / 4;
  const int lane = threadIdx.x & 63;
  const int kk = lane >> 4, jl = lane & 15;
  const int ks = (w + 3) >> 2, rbn = (w + 15) >> 4;
  for (int cc = c0 + 16 * first; cc < c1; cc += 16 * step) {
    cd a[KS];
    {
      const int col = cc + jl;
      const cd* src = M + r0 + (long)col * ld;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int r = 4 * s + kk;
        a[s] = (col < c1 && r < w) ? src[r] : mk(0.0, 0.0);
      }
    }
    // one 16-row block of the result at a time: a[] and one accumulator pair live
    for (int rb = 0; rb < rbn; ++rb) {
      d4 accR = d4{0.0, 0.0, 0.0, 0.0}, accI = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if (s < ks) {
          const cd u = U[4 * s + kk][16 * rb + jl];  // B[k][i] = conj(U[k][i])
          accR = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s].x, u.x, accR, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s].x, -u.y, accI, 0, 0, 0);
          accR = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s].y, u.y, accR, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s].y, u.x, accI, 0, 0, 0);
        }
      }
      // D[j][i] = (U^H M)[i][cc + j], j = kk + 4 q, i = 16 rb + jl
      const int i = 16 * rb + jl;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = cc + kk + 4 * q;
        if (i < w && col < c1) M[(r0 + i) + (long)col * ld] = mk(accR[q], accI[q]);
      }
    }
  }
}

// M[r0:r1, c0:c0+w] <- M[...] U: as D = U^T M^T per 16 rows; the wave takes the 16-row strips
// first, first + step, ..., reads their w columns into registers and writes them back.
template <int W>
__device__ void apply_right_reg(const QMat<W>& U, int w, cd* M, long ld, int r0, int r1, int c0, int first,
                                int step) {
  constexpr int KS = W / 4;
  const int lane = threadIdx.x & 63;
  const int kk = lane >> 4, jl = lane & 15;
  const int ks = (w + 3) >> 2, cbn = (w + 15) >> 4;
  for (int rr = r0 + 16 * first; rr < r1; rr += 16 * step) {
    const int row = rr + jl;
    cd b[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int k = 4 * s + kk;
      b[s] = (row < r1 && k < w) ? M[row + (long)(c0 + k) * ld] : mk(0.0, 0.0);
    }
    for (int cb = 0; cb < cbn; ++cb) {
      d4 accR = d4{0.0, 0.0, 0.0, 0.0}, accI = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        if (s < ks) {
          const cd u = U[4 * s + kk][16 * cb + jl];  // A[j][k] = U[k][j]
          accR = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x, b[s].x, accR, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x, b[s].y, accI, 0, 0, 0);
          accR = __builtin_amdgcn_mfma_f64_16x16x4f64(-u.y, b[s].y, accR, 0, 0, 0);
          accI = __builtin_amdgcn_mfma_f64_16x16x4f64(u.y, b[s].x, accI, 0, 0, 0);
        }
      }
      // D[j][r] = (M U)[rr + r][16 cb + j], j = kk + 4 q, r = jl
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = 16 * cb + kk + 4 * q;
        if (row < r1 && j < w) M[row + (long)(c0 + j) * ld] = mk(accR[q], accI[q]);
      }
    }
  }
}

// Negligible-subdiagonal test (Ahues-Tisseur form) on an LDS block, row k of [l..i].
template <class Mat>
__device__ inline bool negl_lds(const Mat& Hw, int k, int l, int i, double smlnum) {
  const cd hs = Hw[k][k - 1];
  const double ahs = cabs1(hs);
  if (ahs <= smlnum) return true;
  double tst = cabs1(Hw[k - 1][k - 1]) + cabs1(Hw[k][k]);
  if (tst == 0.0) {
    if (k - 2 >= l) tst += cabs1(Hw[k - 1][k - 2]);
    if (k + 1 <= i) tst += cabs1(Hw[k + 1][k]);
  }
  if (ahs <= ULP * tst) {
    const double a1 = ahs, a2 = cabs1(Hw[k - 1][k]);
    const double ab = fmax(a1, a2), ba = fmin(a1, a2);
    const double b1 = cabs1(Hw[k][k]), b2 = cabs1(csub(Hw[k - 1][k - 1], Hw[k][k]));
    const double aa = fmax(b1, b2), bb = fmin(b1, b2);
    const double s = aa + ab;
    if (ba * (ab / s) <= fmax(smlnum, ULP * (bb * (aa / s)))) return true;
  }
  return false;
}

// Complex Givens rotation with real c (LAPACK zlartg semantics):
// [c s; -conj(s) c] [f; g] = [r; 0].
__device__ inline void givens_scaled(cd f, cd g, double& c, cd& s, cd& r) {
  const double f1 = cabsv(f), g1 = cabsv(g);
  if (g1 == 0.0) {
    c = 1.0;
    s = mk(0.0, 0.0);
    r = f;
  } else if (f1 == 0.0) {
    c = 0.0;
    s = cscale(cconj(g), 1.0 / g1);
    r = mk(g1, 0.0);
  } else {
    const double d = hypot(f1, g1);
    const cd ph = cscale(f, 1.0 / f1);
    c = f1 / d;
    s = cscale(cmul(ph, cconj(g)), 1.0 / d);
    r = cscale(ph, d);
  }
}
// One reciprocal square root: with a = 1 / (|f| d), d^2 = |f|^2 + |g|^2, the rotation is
// c = |f|^2 a, s = f conj(g) a, r = f d^2 a. Used when |f|^2 d^2 stays well inside the range.
__device__ __forceinline__ void givens_fast(cd f, cd g, double& c, cd& s, cd& r) {
  const double f2 = cnorm2(f), d2 = f2 + cnorm2(g);
  if (__builtin_expect(!(f2 >= 0x1p-400 && d2 <= 0x1p400), 0)) {
    givens_scaled(f, g, c, s, r);
    return;
  }
  const double a = rsqrt_nr(f2 * d2);
  c = f2 * a;
  s = cscale(cmulc(f, g), a);
  r = cscale(f, d2 * a);
}

// Eigenvalue of the 2x2 block [[a, b], [c, d]] closest to d.
__device__ inline cd wilkinson(cd a, cd b, cd c, cd d) {
  const cd x = cscale(csub(a, d), 0.5), u2 = cmul(b, c);
  const double xx = cnorm2(x), uu = cnorm2(u2);
  if (uu == 0.0 && cabs1(b) * cabs1(c) == 0.0) return d;
  const cd z = cadd(cmul(x, x), u2);
  const double m2 = cnorm2(z);
  // y = sqrt(z) with |z| = sqrt(m2), h = (|Re z| + |z|) / 2, one part sqrt(h), the other Im z / (2 sqrt(h))
  if (xx <= 0x1p200 && uu <= 0x1p400 && m2 >= 0x1p-400) {
    const double h = 0.5 * (fabs(z.x) + m2 * rsqrt_nr(m2));
    const double rh = rsqrt_nr(h);
    const double p = h * rh, q = 0.5 * z.y * rh;
    cd y = z.x >= 0.0 ? mk(p, q) : mk(fabs(q), copysign(p, z.y));
    if (x.x * y.x + x.y * y.y < 0.0) y = cneg(y);
    const cd v = cadd(x, y);
    const double v2 = cnorm2(v);
    if (v2 >= 0x1p-400) return csub(d, cscale(cmulc(u2, v), rcp_nr(v2)));
  }
  const cd u = cmul(csqrt_principal(b), csqrt_principal(c));
  const double su = cabs1(u);
  if (su == 0.0) return d;
  const double sx = cabs1(x);
  const double sc = fmax(su, sx);
  const cd xs = cscale(x, 1.0 / sc), us = cscale(u, 1.0 / sc);
  cd y = cscale(csqrt_principal(cadd(cmul(xs, xs), cmul(us, us))), sc);
  if (sx > 0.0) {
    const cd xn = cscale(x, 1.0 / sx);
    if (xn.x * y.x + xn.y * y.y < 0.0) y = cneg(y);
  }
  return csub(d, cmul(u, cdiv(u, cadd(x, y))));
}

// Orders the LDS accesses of one wavefront: every lane's earlier LDS writes are seen by
// every lane's later reads (LDS executes a wavefront's instructions in order).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// v of lane l (the same l in every lane).
__device__ __forceinline__ double lane_value(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}
__device__ __forceinline__ cd lane_value(cd v, int l) { return mk(lane_value(v.x, l), lane_value(v.y, l)); }
// All LDS reads issued so far have returned (a loop whose body reads registers loaded before
// it would otherwise wait for its own reads at the same place).
__device__ __forceinline__ void lds_wait() { __builtin_amdgcn_s_waitcnt(0xc07f); }
__device__ __forceinline__ cd pick(bool c, cd a, cd b) { return mk(c ? a.x : b.x, c ? a.y : b.y); }

// Complete Schur decomposition of the s x s Hessenberg block in Hw (s <= QW) by
// single-shift QR, run by ONE wavefront, accumulating the transform into U when WU (U must
// hold the identity or an earlier transform). Subdiagonal entries are set to exact zeros on
// deflation, so Hw ends upper triangular. Returns 0 on success, else (index of the
// unconverged eigenvalue + 1).
//
// A sweep is one serial chain of rotations, so the chain alone is kept short: the entries the
// next rotation needs (rows k .. k+2 of columns k, k+1) stay in registers, the same in every
// lane, and never wait for LDS. Row k + 1 as it stands (lane = column) and column k + 1 as it
// stands (lane = row) are carried in registers from step to step, so each step reads one new
// row and one new column, neither of which the chain waits for, and writes one finished row
// and column. HALF (s <= 32): lanes 0..31 rotate the rows of Hw and lanes 32..63 those of U.
// 32 x 32 random blocks: 0.34 us per rotation (about 100 FP64 instructions, issue-bound); with
// the whole step through LDS and a reflector with a square root and two divisions 0.68 us.
template <bool HALF, bool WU, class Mat>
__device__ __forceinline__ int wave_schur_impl(Mat& Hw, Mat& U, int s, int lane) {
  const double smlnum = SAFMIN * ((double)s / ULP);
  const int itmax = 30 * (s > 10 ? s : 10);
  const int col = lane < s ? lane : s - 1;
  const bool ulane = HALF && lane >= 32;
  int row = HALF ? (lane & 31) : lane;
  const bool rowin = row < s;
  if (!rowin) row = s - 1;
  cd* const cr = ulane ? &U[row][0] : &Hw[row][0];  // this lane's row in the column rotations
  // the lane writes column k when k >= cfrom, row k when its column >= k + 2
  const int cfrom = ulane ? ((WU && rowin) ? -1 : 1 << 20) : lane;
  const int rcol = lane < s ? lane : -1;
  int i = s - 1;
  while (i >= 0) {
    int l = 0;
    bool conv = false;
    for (int its = 0; its <= itmax; ++its) {
      wave_sync();
      const bool ng = (lane >= 1 && lane <= i) ? negl_lds(Hw, lane, 0, i, smlnum) : false;
      const unsigned long long mask = __ballot(ng);
      l = mask ? 63 - __clzll(mask) : 0;
      wave_sync();
      if (l > 0 && lane == 0) Hw[l][l - 1] = mk(0.0, 0.0);
      wave_sync();
      if (l >= i) {
        conv = true;
        break;
      }
      cd sh;
      if (its == 10) {
        sh = cadd(Hw[l][l], mk(0.75 * cabs1(Hw[l + 1][l]), 0.0));
      } else if (its == 20) {
        sh = cadd(Hw[i][i], mk(0.75 * cabs1(Hw[i][i - 1]), 0.0));
      } else {
        sh = wilkinson(Hw[i - 1][i - 1], Hw[i - 1][i], Hw[i][i - 1], Hw[i][i]);
      }
      // chain state: (x, y) = column k - 1 of rows k, k + 1; (p, q) = column k of rows k, k + 1
      cd p = Hw[l][l], q = Hw[l + 1][l];
      cd x = csub(p, sh), y = q;
      cd rc = Hw[l][col];  // row k, lane = column (columns > k)
      cd cc = cr[l];       // column k, lane = row (rows < k of Hw; every row of U)
      cd uc = (WU && !HALF) ? U[row][l] : mk(0.0, 0.0);
      lds_wait();
      for (int k = l; k < i; ++k) {
        const cd n = Hw[k + 1][col];
        const cd u = Hw[k + 1][k + 1];
        const cd w = Hw[k + 2 <= i ? k + 2 : i][k + 1];  // below the block: y, q are not used
        const cd b = cr[k + 1];
        const cd ub = (WU && !HALF) ? U[row][k + 1] : mk(0.0, 0.0);
        double c;
        cd sn, r;
        givens_fast(x, y, c, sn, r);
        const cd sc = cconj(sn);
        const cd t = lane_value(rc, k + 1);
        // rows k, k + 1 of columns k, k + 1
        const cd p1 = cadd(cscale(p, c), cmul(sn, q)), q1 = csub(cscale(q, c), cmul(sc, p));
        const cd t1 = cadd(cscale(t, c), cmul(sn, u)), u1 = csub(cscale(u, c), cmul(sc, t));
        // columns k, k + 1 of row k + 1 and of row k + 2 (whose column k is zero)
        x = cadd(cscale(q1, c), cmul(sc, u1));
        p = csub(cscale(u1, c), cmul(sn, q1));
        y = cmul(sc, w);
        q = cscale(w, c);
        // rows k, k + 1 of the columns right of them
        const cd rk = cadd(cscale(rc, c), cmul(sn, n));
        rc = csub(cscale(n, c), cmul(sc, rc));
        // columns k, k + 1 of the rows above (row k enters here) and of U
        const cd a0 = pick(lane == k, p1, cc), b0 = pick(lane == k, t1, b);
        const cd ck = cadd(cscale(a0, c), cmul(sc, b0));
        cc = csub(cscale(b0, c), cmul(sn, a0));
        const bool sub = rcol == (k > l ? k - 1 : -2);  // the subdiagonal entry left behind
        if ((rcol >= k + 2) | sub) Hw[k][lane] = pick(sub, r, rk);
        if (cfrom <= k) cr[k] = ck;
        if (WU && !HALF) {
          const cd uk = cadd(cscale(uc, c), cmul(sc, ub));
          uc = csub(cscale(ub, c), cmul(sn, uc));
          if (rowin) U[row][k] = uk;
        }
        wave_sync();
      }
      if (rcol > i) Hw[i][lane] = rc;
      if (cfrom < i) cr[i] = cc;
      if (WU && !HALF && rowin) U[row][i] = uc;
      if (lane == 0) {
        Hw[i][i] = p;
        Hw[i][i - 1] = x;
      }
    }
    if (!conv) return i + 1;
    i = l - 1;
  }
  wave_sync();
  return 0;
}

template <class Mat>
__device__ __forceinline__ int wave_schur(Mat& Hw, Mat& U, int s, bool wantU, int lane) {
  if (!wantU) return wave_schur_impl<false, false>(Hw, U, s, lane);
  if (s <= 32) return wave_schur_impl<true, true>(Hw, U, s, lane);
  return wave_schur_impl<false, true>(Hw, U, s, lane);
}

// Moves the diagonal entry j of the n x n upper-triangular T up to position to by Givens
// swaps of adjacent entries (LAPACK ztrexc), updating the Schur vectors U (n rows). One
// wavefront, n <= 32: the moving row (lane = column) and the moving column (lane = row; lanes
// 32.. carry U's) stay in registers, as in wave_schur_impl.
template <class Mat>
__device__ __forceinline__ void wave_move_up(Mat& T, Mat& U, int n, int j, int to, int lane) {
  if (j <= to) return;
  const bool ulane = lane >= 32;
  int row = lane & 31;
  const bool rowin = row < n;
  if (!rowin) row = n - 1;
  const int col = lane < n ? lane : n - 1;
  cd* const cr = ulane ? &U[row][0] : &T[row][0];
  const int cfrom = ulane ? (rowin ? -1 : 1 << 20) : lane;  // writes column k + 1 when k >= cfrom
  const int rcol = lane < n ? lane : -1;
  const cd lam = T[j][j];
  const cd dg = T[col][col];  // the diagonal, lane = index
  cd mr = T[j][col];          // the moving row, columns > k + 1
  cd mc = cr[j];              // the moving column, rows <= k (every row of U)
  cd xc = cr[j - 1];          // column k
  wave_sync();
  lds_wait();
  for (int k = j - 1; k >= to; --k) {
    const cd xr = T[k][col];
    const cd xn = cr[k > 0 ? k - 1 : 0];  // the next step's column (this step leaves it alone)
    const cd t11 = lane_value(dg, k);
    const cd g = lane_value(mc, k);  // T[k][k + 1]
    double c;
    cd sn, r;
    givens_fast(g, csub(lam, t11), c, sn, r);
    const cd sc = cconj(sn);
    const cd cdn = pick(lane == k, g, csub(cscale(mc, c), cmul(sn, xc)));  // column k + 1, rows <= k
    mc = cadd(cscale(xc, c), cmul(sc, mc));
    const cd rdn = csub(cscale(mr, c), cmul(sc, xr));  // row k + 1, columns >= k + 2
    mr = pick(lane == k + 1, g, cadd(cscale(xr, c), cmul(sn, mr)));  // T[k][k + 1] keeps its value
    xc = xn;
    wave_sync();
    // row k + 1 from the diagonal on; column k + 1 down to row k (every row of U)
    if (rcol > k) T[k + 1][lane] = pick(lane == k + 1, t11, rdn);
    if (cfrom <= k) cr[k + 1] = cdn;
    wave_sync();
  }
  if (rcol > to) T[to][lane] = mr;
  if (cfrom < to) cr[to] = mc;
  if (lane == 0) T[to][to] = lam;
  wave_sync();
}

// Swap the adjacent diagonal entries k, k+1 of the n x n upper-triangular T (n > 32: one swap
// at a time, through LDS), updating the Schur vectors U (n rows). One wavefront.
template <class Mat>
__device__ __forceinline__ void wave_swap(Mat& T, Mat& U, int n, int k, int lane) {
  const cd t11 = T[k][k], t22 = T[k + 1][k + 1];
  double cs;
  cd sn, r;
  givens_fast(T[k][k + 1], csub(t22, t11), cs, sn, r);
  wave_sync();
  if (lane >= k + 2 && lane < n) {  // rows k, k+1 from column k+2 on
    const cd x = T[k][lane], y = T[k + 1][lane];
    T[k][lane] = cadd(cscale(x, cs), cmul(sn, y));
    T[k + 1][lane] = csub(cscale(y, cs), cmul(cconj(sn), x));
  }
  const cd snc = cconj(sn);
  if (lane < k) {  // columns k, k+1 above row k
    const cd x = T[lane][k], y = T[lane][k + 1];
    T[lane][k] = cadd(cscale(x, cs), cmul(snc, y));
    T[lane][k + 1] = csub(cscale(y, cs), cmul(sn, x));
  }
  if (lane < n) {
    const cd x = U[lane][k], y = U[lane][k + 1];
    U[lane][k] = cadd(cscale(x, cs), cmul(snc, y));
    U[lane][k + 1] = csub(cscale(y, cs), cmul(sn, x));
  }
  if (lane == 0) {
    T[k][k] = t22;
    T[k + 1][k + 1] = t11;
  }
  wave_sync();
}

// T <- G^H T on rows r0..r0+len-1 (columns c0..n-1), then T <- T G on those columns
// (rows 0..rows_t-1) and U <- U G (rows 0..n-1), G = I - tau v v^H with v in vv[0..len).
template <class Mat>
__device__ __forceinline__ void wave_reflect(Mat& T, Mat& U, const cd* vv, cd tau, int r0, int len, int c0, int n,
                                             int rows_t, int lane) {
  // e_q, q < len, at step doubles apart: sum f(v_q) e_q and e_q -= d g(v_q), four at a time
  auto dot = [&](const cd* e, int step, bool conjv) {
    cd d = mk(0.0, 0.0);
    int q = 0;
    for (; q + 4 <= len; q += 4) {
      cd a[4], v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) a[k] = e[(q + k) * step], v[k] = vv[q + k];
#pragma unroll
      for (int k = 0; k < 4; ++k) d = cadd(d, conjv ? cmulc(a[k], v[k]) : cmul(a[k], v[k]));
    }
    for (; q < len; ++q) d = cadd(d, conjv ? cmulc(e[q * step], vv[q]) : cmul(e[q * step], vv[q]));
    return d;
  };
  auto axpy = [&](cd* e, int step, cd d, bool conjv) {
    int q = 0;
    for (; q + 4 <= len; q += 4) {
      cd a[4], v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) a[k] = e[(q + k) * step], v[k] = vv[q + k];
#pragma unroll
      for (int k = 0; k < 4; ++k) e[(q + k) * step] = csub(a[k], conjv ? cmulc(d, v[k]) : cmul(d, v[k]));
    }
    for (; q < len; ++q) e[q * step] = csub(e[q * step], conjv ? cmulc(d, vv[q]) : cmul(d, vv[q]));
  };
  if (lane >= c0 && lane < n) {
    const cd d = cmul(cconj(tau), dot(&T[r0][lane], (int)(&T[1][0] - &T[0][0]), true));
    axpy(&T[r0][lane], (int)(&T[1][0] - &T[0][0]), d, false);
  }
  wave_sync();
  if (n <= 32) {  // lanes 0..31 the rows of T, lanes 32..63 those of U
    const int row = lane & 31;
    if (lane >= 32 ? row < n : row < rows_t) {
      cd* e = lane >= 32 ? &U[row][r0] : &T[row][r0];
      axpy(e, 1, cmul(tau, dot(e, 1, false)), true);
    }
  } else if (lane < n) {
    if (lane < rows_t) axpy(&T[lane][r0], 1, cmul(tau, dot(&T[lane][r0], 1, false)), true);
    axpy(&U[lane][r0], 1, cmul(tau, dot(&U[lane][r0], 1, false)), true);
  }
  wave_sync();
}

// QR kernel configuration: window W, T threads, RA: window products from registers
// (apply_left_reg / apply_right_reg) instead of through an LDS chunk buffer.
// TM: a team of workgroups shares the products (hqr_team_kernel).
template <int W_, int T_, bool RA_, bool TM_ = false>
struct QrCfg {
  static constexpr int W = W_, T = T_;
  static constexpr bool RA = RA_, TM = TM_;
};

template <class C>
__device__ void lds_load_block(QrLds<C::W, C::T>& L, const cd* H, long ldh, int r0, int w) {
  for (int e = threadIdx.x; e < C::W * C::W; e += C::T) {
    const int i = e % C::W, j = e / C::W;
    L.Hw[i][j] = (i < w && j < w) ? H[(r0 + i) + (long)(r0 + j) * ldh] : mk(0.0, 0.0);
    L.U[i][j] = (i == j && i < w) ? mk(1.0, 0.0) : mk(0.0, 0.0);
  }
  __syncthreads();
}

template <class C>
__device__ void lds_store_block(QrLds<C::W, C::T>& L, cd* H, long ldh, int r0, int w) {
  __syncthreads();
  for (int e = threadIdx.x; e < w * w; e += C::T) {
    int i = e % w, j = e / w;
    H[(r0 + i) + (long)(r0 + j) * ldh] = L.Hw[i][j];
  }
  __syncthreads();
}

// Wave gw of nw's share of a window transform U (indices ws..ws+w-1) applied to everything
// outside the window: the rows of the window right of it, its columns above it, and Z. The
// three regions are disjoint; their 16-wide strips are dealt over the waves as one list.
template <int W>
__device__ __forceinline__ void apply_share(const QMat<W>& U, int N, cd* H, long ldh, cd* Z, long ldz, int ws, int w,
                                            int gw, int nw) {
  const int we = ws + w;
  const int nl = (N - we + 15) >> 4, nr = (ws + 15) >> 4;
  apply_left_reg<W>(U, w, H, ldh, ws, we, N, gw, nw);
  apply_right_reg<W>(U, w, H, ldh, 0, ws, ws, (gw + nw - nl % nw) % nw, nw);
  apply_right_reg<W>(U, w, Z, ldz, 0, N, ws, (gw + nw - (nl + nr) % nw) % nw, nw);
}

// A team: the workgroup that iterates on a matrix (the master) and the workgroups that take part
// in its window products. A launch of few matrices leaves most CUs idle while the products of
// one matrix keep one CU's matrix cores busy for two thirds of the iteration. The master
// publishes a window (its transform in global memory and one 64-bit word: sequence number,
// members taking part, window size and start); the members apply their shares and count up
// done. Nobody waits for a workgroup that may not be resident: a member joins only after it
// has seen the master running (or leaves after TEAM_SPINS looks), the master counts only
// members that have joined, and the members leave at the master's last word.
struct TeamCtl {
  unsigned long long word;
  int joined, done;
  int pad[28];  // one line per matrix
};
static_assert(sizeof(TeamCtl) == 128, "team control lines");
constexpr int TEAM_SPINS = 1 << 18;
constexpr unsigned TEAM_EXIT = 0xffffffffu;
constexpr long TEAM_WORK = 150000;  // N w^2 from which a window is shared (measured best of 150000 .. 900000)
struct Team {
  TeamCtl* ctl;
  cd* U;
  unsigned seq;
  int owed;
};
__device__ __forceinline__ unsigned long long team_word(unsigned seq, int members, int w, int ws) {
  return ((unsigned long long)seq << 32) | ((unsigned)members << 24) | ((unsigned)w << 16) | (unsigned)ws;
}
template <class T>
__device__ __forceinline__ T agent_load(T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A workgroup's hand-over: every wave waits until the L2 has its stores (team_drain) before the
// barrier after which one thread writes the L2 back (team_release) and stores the word or counts up
// done. The barrier alone waits for LDS only, so that the one fence would cover its own wave's
// stores and leave those of the other waves to the order inside the CU. The other way round one
// thread invalidates the caches (team_acquire) and waits for that before the barrier. Both fences in
// every wave instead: one matrix stack at N = 882 229 -> 256 ms, 8 at N = 450 137 -> 143 ms.
__device__ __forceinline__ void team_drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void team_release() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent"); }
__device__ __forceinline__ void team_acquire() {
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  team_drain();
}
// One thread, after team_drain() of every wave and a barrier: stores the word.
__device__ __forceinline__ void team_publish(Team& tm, unsigned long long word) {
  team_release();
  __hip_atomic_store(&tm.ctl->word, word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Apply the window transform U (on indices ws..ws+w-1) to everything outside the window. The
// register form needs one barrier at the end only.
template <class C>
__device__ void apply_window(QrLds<C::W, C::T>& L, int N, cd* H, long ldh, cd* Z, long ldz, int ws, int w, Team& tm) {
  const int we = ws + w - 1;
  constexpr int NW = C::T / 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (C::TM) {
    const int t = threadIdx.x;
    int members = 0;
    if ((long)N * w * w >= TEAM_WORK) {
      if (t == 0) L.ctl[3] = agent_load(&tm.ctl->joined);
      __syncthreads();
      members = L.ctl[3];
    }
    if (members > 0) {
      ++tm.seq;
      for (int e = t; e < w * w; e += C::T) tm.U[e] = L.U[e % w][e / w];
      team_drain();
      __syncthreads();
      if (t == 0) team_publish(tm, team_word(tm.seq, members, w, ws));
    }
    apply_share<C::W>(L.U, N, H, ldh, Z, ldz, ws, w, wave, NW * (members + 1));
    __syncthreads();
    if (members > 0) {
      tm.owed += members;
      if (t == 0) {
        while (agent_load(&tm.ctl->done) < tm.owed) __builtin_amdgcn_s_sleep(1);
        team_acquire();
      }
      __syncthreads();
    }
  } else if constexpr (C::RA) {
    apply_share<C::W>(L.U, N, H, ldh, Z, ldz, ws, w, wave, NW);
    __syncthreads();
  } else {
    static_assert(C::W == QW && C::T == QT, "the LDS-staged window products are written for W = 64, 512 threads");
    if (we + 1 < N) apply_left_u(L.U, L.Hw, w, H, ldh, ws, we + 1, N);
    if (ws > 0) apply_right_u(L.U, L.Hw, w, H, ldh, 0, ws, ws);
    apply_right_u(L.U, L.Hw, w, Z, ldz, 0, N, ws);
  }
}

// A team member's whole run: join, then take part in every published window that counts it.
template <class C>
__device__ void team_member(QrLds<C::W, C::T>& L, int N, cd* H, long ldh, cd* Z, long ldz, Team tm) {
  constexpr int NW = C::T / 64;
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  unsigned seen = 0;
  if (t == 0) {
    int k = 0;
    for (int spin = 0; spin < TEAM_SPINS; ++spin) {
      seen = (unsigned)(agent_load(&tm.ctl->word) >> 32);
      if (seen != 0) break;
      __builtin_amdgcn_s_sleep(8);
    }
    if (seen != 0 && seen != TEAM_EXIT)
      k = 1 + __hip_atomic_fetch_add(&tm.ctl->joined, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    L.ctl[0] = k;
  }
  __syncthreads();
  const int k = L.ctl[0];
  if (k == 0) return;
  for (;;) {
    __syncthreads();
    if (t == 0) {
      unsigned long long word = agent_load(&tm.ctl->word);
      while ((unsigned)(word >> 32) == seen) {
        __builtin_amdgcn_s_sleep(2);
        word = agent_load(&tm.ctl->word);
      }
      seen = (unsigned)(word >> 32);
      team_acquire();
      L.ctl[1] = seen == TEAM_EXIT ? 1 : 0;
      L.ctl[2] = (int)(unsigned)(word & 0xffffffffu);
    }
    __syncthreads();
    if (L.ctl[1]) return;
    const unsigned par = (unsigned)L.ctl[2];
    const int members = (int)(par >> 24), w = (int)((par >> 16) & 0xff), ws = (int)(par & 0xffff);
    if (members < k) continue;  // published before this member joined
    for (int e = t; e < C::W * C::W; e += C::T) {
      const int i = e % C::W, j = e / C::W;
      L.U[i][j] = (i < w && j < w) ? tm.U[i + j * w] : mk(0.0, 0.0);
    }
    __syncthreads();
    apply_share<C::W>(L.U, N, H, ldh, Z, ldz, ws, w, k * NW + wave, NW * (members + 1));
    team_drain();
    __syncthreads();
    if (t == 0) {
      team_release();
      __hip_atomic_fetch_add(&tm.ctl->done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// Aggressive early deflation (the deflation-window step of LAPACK zlaqr3) on the
// trailing nw x nw window of the active block [lo, hi]: Schur form of the window,
// spike deflation test with reordering of the undeflatable eigenvalues to the top,
// re-reduction of the undeflated part to Hessenberg form, and the window transform
// applied to the rest of H and to Z. Returns the number of deflated eigenvalues (-1 if
// the window's QR did not converge; nothing is changed then). The undeflated
// eigenvalues are left in L.aedv[0..*nsa) for use as shifts.
template <class C>
__device__ int aed(QrLds<C::W, C::T>& L, int N, cd* H, long ldh, cd* Z, long ldz, int lo, int hi, int nw,
                    int* nsa, Team& tm) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int kwtop = hi - nw + 1;
  const cd spike = (kwtop > lo) ? H[kwtop + (long)(kwtop - 1) * ldh] : mk(0.0, 0.0);
  lds_load_block<C>(L, H, ldh, kwtop, nw);
  if (wave == 0) {
    const int info = wave_schur(L.Hw, L.U, nw, true, lane);
    if (lane == 0) L.ctl[1] = info;
    if (info == 0) {
      auto& T = L.Hw;
      auto& U = L.U;
      const double smlnum = SAFMIN * ((double)N / ULP);
      const double as = cabs1(spike);
      int ns = nw, ilst = 0;
      for (int knt = 0; knt < nw; ++knt) {
        const int j = ns - 1;
        double foo = cabs1(T[j][j]);
        if (foo == 0.0) foo = as;
        const bool defl = as * cabs1(U[0][j]) <= fmax(smlnum, ULP * foo);
        wave_sync();
        if (defl) {
          --ns;
        } else {
          if (nw <= 32)
            wave_move_up(T, U, nw, j, ilst, lane);
          else
            for (int k = j - 1; k >= ilst; --k) wave_swap(T, U, nw, k, lane);
          ++ilst;
        }
      }
      if (lane < ns) L.aedv[lane] = T[lane][lane];
      wave_sync();
      cd newspike = mk(0.0, 0.0);
      if (ns > 0 && (spike.x != 0.0 || spike.y != 0.0)) {
        // shifts are kept in ctl-free storage: copy the undeflated eigenvalues first
        cd ev = lane < ns ? L.aedv[lane] : mk(0.0, 0.0);
        if (ns > 1) {
          // reflect the spike s * conj(U[0][0..ns)) onto e1 (zlaqr3 "reflect spike back")
          cd w = lane < ns ? cconj(U[0][lane]) : mk(0.0, 0.0);
          const cd alpha = cconj(U[0][0]);
          double beta;
          cd tau, scale;
          wave_house(alpha, lane >= 1 && lane < ns ? w : mk(0.0, 0.0), beta, tau, scale);
          wave_sync();
          L.aedv[lane] = lane == 0 ? mk(1.0, 0.0) : (lane < ns ? cmul(w, scale) : mk(0.0, 0.0));
          wave_sync();
          wave_reflect(T, U, L.aedv, tau, 0, ns, 0, nw, ns, lane);
          // Hessenberg reduction of T[0:ns, 0:ns] (columns 0..ns-3)
          for (int c = 0; c + 2 < ns; ++c) {
            const int len = ns - c - 1;
            const cd a0 = T[c + 1][c];
            const cd xv = (lane >= c + 2 && lane < ns) ? T[lane][c] : mk(0.0, 0.0);
            double bc;
            cd tc, sc;
            wave_house(a0, xv, bc, tc, sc);
            wave_sync();
            if (lane < len) L.aedv[lane] = lane == 0 ? mk(1.0, 0.0) : cmul(T[c + 1 + lane][c], sc);
            wave_sync();
            if (lane == c) {
              T[c + 1][c] = mk(bc, 0.0);
              for (int r = c + 2; r < ns; ++r) T[r][c] = mk(0.0, 0.0);
            }
            wave_sync();
            if (tc.x != 0.0 || tc.y != 0.0) wave_reflect(T, U, L.aedv, tc, c + 1, len, c + 1, nw, ns, lane);
          }
        }
        newspike = cmul(spike, cconj(U[0][0]));
        wave_sync();
        if (lane < ns) L.aedv[lane] = ev;  // shifts for the next sweep
        wave_sync();
      }
      if (lane == 0) {
        L.ctl[2] = ns;
        L.shifts[0] = newspike;  // staging; read back before the next use of shifts
      }
    }
  }
  __syncthreads();
  if (L.ctl[1] != 0) {
    __syncthreads();
    *nsa = 0;
    return -1;
  }
  const int ns = L.ctl[2];
  const cd newspike = L.shifts[0];
  __syncthreads();
  lds_store_block<C>(L, H, ldh, kwtop, nw);
  if (t == 0 && kwtop > lo) H[kwtop + (long)(kwtop - 1) * ldh] = newspike;
  __syncthreads();
  apply_window<C>(L, N, H, ldh, Z, ldz, kwtop, nw, tm);
  *nsa = ns;
  return nw - ns;
}

// Largest k in [1, hi] whose subdiagonal is negligible (sets it to zero); 0 if none.
template <class C>
__device__ int find_lo(QrLds<C::W, C::T>& L, cd* H, long ldh, int N, int hi) {
  const int t = threadIdx.x;
  const double smlnum = SAFMIN * ((double)N / ULP);
  int best = 0;
  for (int k = hi - t; k >= 1; k -= C::T) {
    const cd hs = H[k + (long)(k - 1) * ldh];
    const double ahs = cabs1(hs);
    bool ng = ahs <= smlnum;
    if (!ng) {
      const cd hkk = H[k + (long)k * ldh], hk1 = H[(k - 1) + (long)(k - 1) * ldh];
      double tst = cabs1(hk1) + cabs1(hkk);
      if (tst == 0.0) {
        if (k >= 2) tst += cabs1(H[(k - 1) + (long)(k - 2) * ldh]);
        if (k + 1 <= hi) tst += cabs1(H[(k + 1) + (long)k * ldh]);
      }
      if (ahs <= ULP * tst) {
        const double a2 = cabs1(H[(k - 1) + (long)k * ldh]);
        const double ab = fmax(ahs, a2), ba = fmin(ahs, a2);
        const double b1 = cabs1(hkk), b2 = cabs1(csub(hk1, hkk));
        const double aa = fmax(b1, b2), bb = fmin(b1, b2);
        const double s = aa + ab;
        ng = ba * (ab / s) <= fmax(smlnum, ULP * (bb * (aa / s)));
      }
    }
    if (ng) {
      best = k;
      break;
    }
  }
  L.redi[t] = best;
  __syncthreads();
  for (int w = C::T / 2; w > 0; w >>= 1) {
    if (t < w && L.redi[t + w] > L.redi[t]) L.redi[t] = L.redi[t + w];
    __syncthreads();
  }
  const int lo = L.redi[0];
  __syncthreads();
  if (t == 0 && lo > 0) H[lo + (long)(lo - 1) * ldh] = mk(0.0, 0.0);
  __syncthreads();
  return lo;
}

// A bulge of the chase, owned by one wave for a whole window. The reflector (v1, v2, tau)
// stays in the wave's registers between the row and the column operations of a step, and
// the two columns of U that the next step touches again (u0, u1) stay there between steps:
// the step then reads one column of U and writes one. LDS bandwidth bounds the chase (three
// rows and three columns of the window read and written per bulge and step).
struct Bulge {
  cd v1, v2, tau;
  cd u0, u1;
};
struct ChasePos {
  int lo, hi, ws, w, t0, t1;
};

// The step's reflectors from the bulges' three entries (columns left of the bulge are zero)
// applied to their rows, lane = column. Bulges NJ at once (b[m], index bb[m]), so that one's
// dependency chain hides the other's; the rows of different bulges are disjoint, so the waves
// need no barrier here.
template <class C, int NJ>
__device__ __forceinline__ void chase_rows(QrLds<C::W, C::T>& L, const ChasePos& cp, int tt, Bulge* const (&b)[NJ],
                                           const int (&bb)[NJ], int lane) {
  cd h1[NJ], h2[NJ], h3[NJ], e1[NJ], e2[NJ], e3[NJ];
#pragma unroll
  for (int m = 0; m < NJ; ++m) {
    const int p = cp.lo - 1 + tt - 3 * bb[m];
    const int r1 = p + 1 - cp.ws, r3 = r1 + (p + 3 <= cp.hi ? 2 : 1);
    const int j0 = r1 > 0 ? r1 - 1 : 0, j = j0 + lane;
    const int jc = j < cp.w ? j : cp.w - 1;
    h1[m] = L.Hw[r1][jc];
    h2[m] = L.Hw[r1 + 1][jc];
    h3[m] = L.Hw[r3][jc];
    e1[m] = L.Hw[r1][j0];
    e2[m] = L.Hw[r1 + 1][j0];
    e3[m] = L.Hw[r3][j0];
  }
#pragma unroll
  for (int m = 0; m < NJ; ++m) {
    const int p = cp.lo - 1 + tt - 3 * bb[m];
    const bool three = p + 3 <= cp.hi, fresh = p == cp.lo - 1;
    const int r1 = p + 1 - cp.ws;
    const int j = (r1 > 0 ? r1 - 1 : 0) + lane;
    cd x = e1[m], y = e2[m], z = e3[m];
    if (fresh) {  // a new bulge: the first column of (H - s1)(H - s2); lane 0 holds column lo
      const cd s1 = L.shifts[2 * bb[m]], s2 = L.shifts[2 * bb[m] + 1];
      const cd h11 = x, h21 = y, h12 = lane_value(h1[m], 1), h22 = lane_value(h2[m], 1), h32 = lane_value(h3[m], 1);
      const double sc = cabs1(csub(h11, s2)) + cabs1(h21);
      if (sc == 0.0) {
        x = y = z = mk(0.0, 0.0);
      } else {
        const cd h21s = cscale(h21, 1.0 / sc);
        x = cadd(cmul(h21s, h12), cmul(csub(h11, s1), cscale(csub(h11, s2), 1.0 / sc)));
        y = cmul(h21s, csub(cadd(h11, h22), cadd(s1, s2)));
        z = cmul(h21s, h32);
      }
    }
    if (!three) z = h3[m] = mk(0.0, 0.0);
    double beta;
    cd tau, scale;
    house_small(x, y, z, beta, tau, scale);
    const cd v1 = cmul(y, scale), v2 = cmul(z, scale);
    b[m]->v1 = v1;
    b[m]->v2 = v2;
    b[m]->tau = tau;
    const cd sm = cmul(cconj(tau), cadd(cadd(h1[m], cmulc(h2[m], v1)), cmulc(h3[m], v2)));
    // the bulge's own column (absent for a new bulge) becomes (beta, 0, 0)
    const bool own = !fresh && lane == 0;
    const cd o1 = pick(own, mk(beta, 0.0), csub(h1[m], sm));
    const cd o2 = pick(own, mk(0.0, 0.0), csub(h2[m], cmul(sm, v1)));
    const cd o3 = pick(own, mk(0.0, 0.0), csub(h3[m], cmul(sm, v2)));
    if (j < cp.w) {
      L.Hw[r1][j] = o1;
      L.Hw[r1 + 1][j] = o2;
      if (three) L.Hw[r1 + 2][j] = o3;
    }
  }
}

// The same reflectors on the columns of the window (rows down to the bulge's last row + 1;
// below it the columns hold exact zeros) and on those of U, lane = row.
template <class C, int NJ>
__device__ __forceinline__ void chase_cols(QrLds<C::W, C::T>& L, const ChasePos& cp, int tt, Bulge* const (&b)[NJ],
                                           const int (&bb)[NJ], int lane) {
  cd c1[NJ], c2[NJ], c3[NJ], u3[NJ];
  const int row = lane < cp.w ? lane : cp.w - 1;
#pragma unroll
  for (int m = 0; m < NJ; ++m) {
    const int p = cp.lo - 1 + tt - 3 * bb[m];
    const int r1 = p + 1 - cp.ws, r3 = r1 + (p + 3 <= cp.hi ? 2 : 1);
    c1[m] = L.Hw[row][r1];
    c2[m] = L.Hw[row][r1 + 1];
    c3[m] = L.Hw[row][r3];
    u3[m] = L.U[row][r3];
    if (tt == cp.t0 || p == cp.lo - 1) {  // the bulge's first step in this window
      b[m]->u0 = L.U[row][r1];
      b[m]->u1 = L.U[row][r1 + 1];
    }
  }
#pragma unroll
  for (int m = 0; m < NJ; ++m) {
    const int p = cp.lo - 1 + tt - 3 * bb[m];
    const bool three = p + 3 <= cp.hi;
    const int r1 = p + 1 - cp.ws;
    const cd v1 = b[m]->v1, v2 = b[m]->v2, tau = b[m]->tau;
    if (!three) c3[m] = u3[m] = mk(0.0, 0.0);
    const cd sm = cmul(tau, cadd(cadd(c1[m], cmul(c2[m], v1)), cmul(c3[m], v2)));
    const cd su = cmul(tau, cadd(cadd(b[m]->u0, cmul(b[m]->u1, v1)), cmul(u3[m], v2)));
    const cd w0 = csub(b[m]->u0, su), w1 = csub(b[m]->u1, cmulc(su, v1)), w2 = csub(u3[m], cmulc(su, v2));
    const cd o1 = csub(c1[m], sm), o2 = csub(c2[m], cmulc(sm, v1)), o3 = csub(c3[m], cmulc(sm, v2));
    b[m]->u0 = w1;
    b[m]->u1 = w2;
    if (lane < cp.w) {
      L.U[row][r1] = w0;
      if (!three) {
        L.U[row][r1 + 1] = w1;
      } else if (tt == cp.t1 - 1) {  // leaving the window
        L.U[row][r1 + 1] = w1;
        L.U[row][r1 + 2] = w2;
      }
      if (lane <= r1 + 3) {
        L.Hw[row][r1] = o1;
        L.Hw[row][r1 + 1] = o2;
        if (three) L.Hw[row][r1 + 2] = o3;
      }
    }
  }
}

// One multishift sweep over the active block [lo, hi] with nbul bulges (shifts in L.shifts);
// wave v owns the bulges v, v + T/64, ... A chase step has two barriers: after the rows and
// after the columns.
template <class C>
__device__ void qr_sweep(QrLds<C::W, C::T>& L, int N, cd* H, long ldh, cd* Z, long ldz, int lo, int hi, int nbul,
                         long long* st, Team& tm) {
  constexpr int NW = C::T / 64;
  constexpr int MB = ((C::W - 9) / 3 < NBUL ? (C::W - 9) / 3 : NBUL) / NW + 1 & ~1;  // bulges per wave, even
  static_assert(MB * NW >= ((C::W - 9) / 3 < NBUL ? (C::W - 9) / 3 : NBUL), "every bulge has a wave");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int adv = C::W - 3 * nbul - 1;
  const int T_end = (hi - 2) - (lo - 1) + 3 * (nbul - 1) + 1;
  for (int t0 = 0; t0 < T_end; t0 += adv) {
    const int t1 = t0 + adv < T_end ? t0 + adv : T_end;
    int pmin = lo - 1 + t0 - 3 * (nbul - 1);
    if (pmin < lo - 1) pmin = lo - 1;
    int pmax = lo - 1 + t1 - 1;
    if (pmax > hi - 2) pmax = hi - 2;
    const int ws = pmin > lo ? pmin : lo;
    const int we = pmax + 4 < hi ? pmax + 4 : hi;
    const int w = we - ws + 1;
    const long long c0 = wall_clock64();
    lds_load_block<C>(L, H, ldh, ws, w);
    const ChasePos cp = {lo, hi, ws, w, t0, t1};
    Bulge bul[MB];
    for (int tt = t0; tt < t1; ++tt) {
      // bulge bb is active when lo - 1 <= p <= hi - 2, p = lo - 1 + tt - 3 bb
      auto active = [&](int bb) { return bb < nbul && tt >= 3 * bb && lo - 1 + tt - 3 * bb <= hi - 2; };
#pragma unroll
      for (int m = 0; m < MB; m += 2) {
        const int b0 = wave + m * NW, b1 = b0 + NW;
        const bool a0 = active(b0), a1 = active(b1);
        if (a0 && a1)
          chase_rows<C, 2>(L, cp, tt, {&bul[m], &bul[m + 1]}, {b0, b1}, lane);
        else if (a0)
          chase_rows<C, 1>(L, cp, tt, {&bul[m]}, {b0}, lane);
        else if (a1)
          chase_rows<C, 1>(L, cp, tt, {&bul[m + 1]}, {b1}, lane);
      }
      __syncthreads();
#pragma unroll
      for (int m = 0; m < MB; m += 2) {
        const int b0 = wave + m * NW, b1 = b0 + NW;
        const bool a0 = active(b0), a1 = active(b1);
        if (a0 && a1)
          chase_cols<C, 2>(L, cp, tt, {&bul[m], &bul[m + 1]}, {b0, b1}, lane);
        else if (a0)
          chase_cols<C, 1>(L, cp, tt, {&bul[m]}, {b0}, lane);
        else if (a1)
          chase_cols<C, 1>(L, cp, tt, {&bul[m + 1]}, {b1}, lane);
      }
      __syncthreads();
    }
    lds_store_block<C>(L, H, ldh, ws, w);
    const long long c1 = wall_clock64();
    apply_window<C>(L, N, H, ldh, Z, ldz, ws, w, tm);
    const long long c2 = wall_clock64();
    st[1] += 1;
    st[2] += c1 - c0;
    st[3] += c2 - c1;
  }
}

// stats (nullable): per matrix {sweeps, windows, window-chase ticks, off-window-apply ticks,
// small-block ticks} of the constant-rate device clock.
// use_aed: deflation-window size (0 = no aggressive early deflation); max_bul: bulges
// per sweep (<= NBUL).
template <class C>
__device__ void hqr_body(QrLds<C::W, C::T>& L, int N, cd* H, long ldh, long sH, cd* Z, long ldz, long sZ, cd* wout,
                         long sw, int* info, long long* stats, int use_aed, int max_bul, int max_sweeps, long b,
                         Team tm) {
  long long st[5] = {0, 0, 0, 0, 0};
  H += b * sH;
  Z += b * sZ;
  wout += b * sw;
  const int t = threadIdx.x;
  // blocks this small are finished by the single-wave QR in the window; at least 8 chase
  // steps per window
  constexpr int NMIN = QR_NMIN < C::W ? QR_NMIN : C::W;
  constexpr int BMAX = (C::W - 9) / 3 < NBUL ? (C::W - 9) / 3 : NBUL;
  if (max_bul > BMAX) max_bul = BMAX;
  if (use_aed > C::W - 1) use_aed = C::W - 1;
  int ihi = N - 1;
  int sweeps = 0, last_progress = 0, prev_lo = -1, prev_hi = N;
  const int itmax = max_sweeps > 0 ? max_sweeps : 30 * (N > 10 ? N : 10);
  int fail = 0;
  while (ihi >= 0) {
    const int lo = find_lo<C>(L, H, ldh, N, ihi);
    const int m = ihi - lo + 1;
    if (lo != prev_lo || ihi != prev_hi) last_progress = sweeps;
    prev_lo = lo;
    prev_hi = ihi;
    if (m <= NMIN) {
      const long long c0 = wall_clock64();
      lds_load_block<C>(L, H, ldh, lo, m);
      if ((t >> 6) == 0) {
        const int r = wave_schur(L.Hw, L.U, m, true, t & 63);
        if (t == 0) L.ctl[1] = r;
      }
      __syncthreads();
      const int r = L.ctl[1];
      lds_store_block<C>(L, H, ldh, lo, m);
      if (r != 0) {
        fail = lo + r;
        break;
      }
      apply_window<C>(L, N, H, ldh, Z, ldz, lo, m, tm);
      st[4] += wall_clock64() - c0;
      ihi = lo - 1;
      continue;
    }
    if (sweeps >= itmax) {
      fail = ihi + 1;
      break;
    }
    int nbul = (m - 2) / 6;
    if (nbul > max_bul) nbul = max_bul;
    if (nbul < 1) nbul = 1;
    // aggressive early deflation on the trailing window
    int nsa = 0;
    if (use_aed) {
      const long long c0 = wall_clock64();
      const int nw = m - 1 < use_aed ? m - 1 : use_aed;
      const int nd = aed<C>(L, N, H, ldh, Z, ldz, lo, ihi, nw, &nsa, tm);
      st[4] += wall_clock64() - c0;
      if (nd > 0) {
        ihi -= nd;
        last_progress = sweeps;
        prev_hi = ihi;
        // a productive window: look again before sweeping (LAPACK's nibble rule)
        if (100 * nd > AED_NIBBLE * nw || ihi - lo + 1 <= NMIN) {
          ++sweeps;
          continue;
        }
      }
      if (nd < 0) nsa = 0;
      const int mm = ihi - lo + 1;
      nbul = (mm - 2) / 6;
      if (nbul > max_bul) nbul = max_bul;
      if (nbul < 1) nbul = 1;
    }
    int ns = 2 * nbul;
    const bool exceptional = (sweeps - last_progress) > 0 && ((sweeps - last_progress) % EXC_SWEEPS) == 0;
    if (exceptional) {
      if (t < ns) {
        const int k = ihi - t;
        cd hk = H[k + (long)k * ldh];
        double sub = cabs1(H[k + (long)(k - 1) * ldh]);
        L.shifts[t] = cadd(hk, mk(0.75 * sub, 0.0));
      }
      __syncthreads();
    } else if (nsa >= 2) {
      // the undeflated window eigenvalues nearest the bottom serve as shifts
      if (nsa < ns) {
        nbul = nsa / 2 > 0 ? nsa / 2 : 1;
        ns = 2 * nbul;
      }
      if (t < ns) L.shifts[t] = L.aedv[nsa - ns + t];
      __syncthreads();
    } else {
      const int r0 = ihi - ns + 1;
      for (int e = t; e < C::W * C::W; e += C::T) {
        const int i = e % C::W, j = e / C::W;
        L.Hw[i][j] = (i < ns && j < ns) ? H[(r0 + i) + (long)(r0 + j) * ldh] : mk(0.0, 0.0);
      }
      __syncthreads();
      if ((t >> 6) == 0) wave_schur(L.Hw, L.U, ns, false, t & 63);
      __syncthreads();
      if (t < ns) L.shifts[t] = L.Hw[t][t];
      __syncthreads();
    }
    qr_sweep<C>(L, N, H, ldh, Z, ldz, lo, ihi, nbul, st, tm);
    ++sweeps;
  }
  __syncthreads();
  if (C::TM && t == 0) team_publish(tm, team_word(TEAM_EXIT, 0, 0, 0));
  for (int i = t; i < N; i += C::T) wout[i] = H[i + (long)i * ldh];
  if (t == 0) {
    info[b] = fail;
    if (stats) {
      st[0] = sweeps;
      for (int k = 0; k < 5; ++k) stats[b * 5 + k] = st[k];
    }
  }
}

// Kernels of the three configurations (one workgroup per matrix): W = 64 on 512 threads with
// the register (hqr_kernel) or the LDS-staged (hqr_lds_kernel) window products, and W = 48
// on 256 threads, two workgroups per CU (at most 256 VGPRs per lane).
#define HQR_ARGS                                                                                       \
  int N, cd *H, long ldh, long sH, cd *Z, long ldz, long sZ, cd *wout, long sw, int *info, long long *stats, \
      int use_aed, int max_bul, int max_sweeps
#define HQR_PASS \
  N, H, ldh, sH, Z, ldz, sZ, wout, sw, info, stats, use_aed, max_bul, max_sweeps, (long)blockIdx.x, Team{}
__global__ __launch_bounds__(512) void hqr_kernel(HQR_ARGS) {
  __shared__ QrLds<64, 512> L;
  hqr_body<QrCfg<64, 512, true>>(L, HQR_PASS);
}
__global__ __launch_bounds__(512) void hqr_lds_kernel(HQR_ARGS) {
  __shared__ QrLds<64, 512> L;
  hqr_body<QrCfg<64, 512, false>>(L, HQR_PASS);
}
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void hqr_w48_kernel(HQR_ARGS) {
  __shared__ QrLds<48, 256> L;
  hqr_body<QrCfg<48, 256, true>>(L, HQR_PASS);
}
// W = 32 on 128 threads: four workgroups (matrices) per CU, for small N.
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2))) void hqr_w32_kernel(HQR_ARGS) {
  __shared__ QrLds<32, 128> L;
  hqr_body<QrCfg<32, 128, true>>(L, HQR_PASS);
}
// The W = 64 kernel with a team of workgroups per matrix, for launches that leave CUs idle.
// Workgroup i < batch is the master of matrix i; the members of matrix b follow at the ids
// that keep the team on the master's XCD (workgroups go to the 8 XCDs in turn), so its
// windows pass through one L2. batch8: the batch rounded up to whole rounds of 8. QR stage of
// 10 matrices at N = 882 with teams of 16: 305 -> 137 ms (the products 193 -> 25 ms), of 80 at
// N = 450 with teams of 3: 77.5 -> 62.7 ms, of 91 at N = 270 with teams of 2: 29.6 -> 25.4 ms.
__global__ __launch_bounds__(512) void hqr_team_kernel(HQR_ARGS, int batch, int batch8, TeamCtl* ctl, cd* Uteam) {
  __shared__ QrLds<64, 512> L;
  typedef QrCfg<64, 512, true, true> C;
  const int id = blockIdx.x, b = id % batch8;
  if (b >= batch) return;
  Team tm = {ctl + b, Uteam + (long)b * QW * QW, 1u, 0};
  if (id >= batch8) {
    team_member<C>(L, N, H + b * sH, ldh, Z + b * sZ, ldz, tm);
    return;
  }
  if (threadIdx.x == 0) team_publish(tm, team_word(1u, 0, 0, 0));
  hqr_body<C>(L, N, H, ldh, sH, Z, ldz, sZ, wout, sw, info, stats, use_aed, max_bul, max_sweeps, (long)b, tm);
}
#undef HQR_ARGS
#undef HQR_PASS

// ===================================================================== eigenvectors
// X (n x n, pre-zeroed) <- upper-triangular eigenvector matrix of upper-triangular T:
// (T - T_kk I) x_k = 0, x_k(k) = 1, tiny pivots replaced by smin (LAPACK ztrevc rule).
__global__ __launch_bounds__(256) void trevc_kernel(int N, const cd* T, long ldt, long sT, cd* X, long ldx,
                                                    long sX) {
  __shared__ LdsMat Ts;
  __shared__ LdsMat Xs;
  __shared__ cd lam[QW];
  __shared__ double smin[QW];
  const long b = blockIdx.y;
  T += b * sT;
  X += b * sX;
  const int K = blockIdx.x;
  const int k0 = K * QW;
  const int bk = N - k0 < QW ? N - k0 : QW;
  const int t = threadIdx.x;
  for (int e = t; e < QW * QW; e += 256) {
    int i = e & 63, j = e >> 6;
    Ts[i][j] = (i < bk && j < bk) ? T[(k0 + i) + (long)(k0 + j) * ldt] : mk(0.0, 0.0);
  }
  __syncthreads();
  if (t < bk) {
    lam[t] = Ts[t][t];
    smin[t] = fmax(ULP * cabs1(lam[t]), SAFMIN * ((double)N / ULP));
  }
  __syncthreads();
  // diagonal tile: thread c solves its own column
  if (t < QW) {
    const int c = t;
    for (int i = 0; i < QW; ++i) Xs[i][c] = mk(0.0, 0.0);
    if (c < bk) {
      Xs[c][c] = mk(1.0, 0.0);
      for (int i = c - 1; i >= 0; --i) {
        cd s = mk(0.0, 0.0);
        for (int j = i + 1; j <= c; ++j) s = cadd(s, cmul(Ts[i][j], Xs[j][c]));
        cd d = csub(Ts[i][i], lam[c]);
        if (cabs1(d) < smin[c]) d = mk(smin[c], 0.0);
        Xs[i][c] = cneg(cdiv(s, d));
      }
    }
  }
  __syncthreads();
  for (int e = t; e < bk * bk; e += 256) {
    int i = e % bk, j = e / bk;
    X[(k0 + i) + (long)(k0 + j) * ldx] = Xs[i][j];
  }
  // right-hand sides for the rows above: X[0:k0, K] = -T[0:k0, K] * X_KK
  for (int rr = 0; rr < k0; rr += QW) {
    __syncthreads();
    for (int e = t; e < QW * QW; e += 256) {
      int i = e & 63, k = e >> 6;
      Ts[i][k] = (k < bk) ? T[(rr + i) + (long)(k0 + k) * ldt] : mk(0.0, 0.0);
    }
    __syncthreads();
    d4 aR[2][2], aI[2][2];
    mm64<false>(Ts, Xs, QW / 4, aR, aI);
    mm64_for_each(aR, aI, [&](int i, int j, cd v) {
      if (j < bk) X[(rr + i) + (long)(k0 + j) * ldx] = cneg(v);
    });
  }
  // block back-substitution upward
  for (int I = K - 1; I >= 0; --I) {
    const int i0 = I * QW;
    __syncthreads();
    for (int e = t; e < QW * QW; e += 256) {
      int i = e & 63, j = e >> 6;
      Ts[i][j] = T[(i0 + i) + (long)(i0 + j) * ldt];
      Xs[i][j] = (j < bk) ? X[(i0 + i) + (long)(k0 + j) * ldx] : mk(0.0, 0.0);
    }
    __syncthreads();
    if (t < bk) {
      const int c = t;
      for (int i = QW - 1; i >= 0; --i) {
        cd s = Xs[i][c];
        for (int j = i + 1; j < QW; ++j) s = csub(s, cmul(Ts[i][j], Xs[j][c]));
        cd d = csub(Ts[i][i], lam[c]);
        if (cabs1(d) < smin[c]) d = mk(smin[c], 0.0);
        Xs[i][c] = cdiv(s, d);
      }
    }
    __syncthreads();
    for (int e = t; e < QW * bk; e += 256) {
      int i = e & 63, j = e >> 6;
      X[(i0 + i) + (long)(k0 + j) * ldx] = Xs[i][j];
    }
    for (int rr = 0; rr < i0; rr += QW) {
      __syncthreads();
      for (int e = t; e < QW * QW; e += 256) {
        int i = e & 63, k = e >> 6;
        Ts[i][k] = T[(rr + i) + (long)(i0 + k) * ldt];
      }
      __syncthreads();
      d4 aR[2][2], aI[2][2];
      mm64<false>(Ts, Xs, QW / 4, aR, aI);
      mm64_for_each(aR, aI, [&](int i, int j, cd v) {
        if (j < bk) {
          cd* p = X + (rr + i) + (long)(k0 + j) * ldx;
          *p = csub(*p, v);
        }
      });
    }
  }
}

// Unit 2-norm, then rotate so that the largest-modulus component (first on ties) is real.
__global__ __launch_bounds__(256) void normalize_cols_kernel(int N, cd* V, long ldv, long sV) {
  const long b = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = blockIdx.x * 4 + wave;
  if (col >= N) return;
  cd* v = V + b * sV + (long)col * ldv;
  double ss = 0.0;
  for (int r = lane; r < N; r += 64) ss += cnorm2(v[r]);
  ss = wsum(ss);
  const double scl = 1.0 / sqrt(ss);
  double best = -1.0;
  int bi = 0x7fffffff;
  for (int r = lane; r < N; r += 64) {
    cd x = cscale(v[r], scl);
    double m = cnorm2(x);
    if (m > best) { best = m; bi = r; }
  }
  for (int o = 32; o > 0; o >>= 1) {
    double ob = __shfl_xor(best, o, 64);
    int oi = __shfl_xor(bi, o, 64);
    if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
  }
  if (bi >= N) bi = 0;  // no component compares (NaN): the vector stays NaN
  const cd vk = cscale(v[bi], scl);
  const cd rot = cscale(cconj(vk), 1.0 / sqrt(best));
  for (int r = lane; r < N; r += 64) {
    cd x = cmul(cscale(v[r], scl), rot);
    if (r == bi) x.y = 0.0;
    v[r] = x;
  }
}

// ===================================================================== balancing
// Diagonal similarity scaling by powers of two (the scaling half of LAPACK zgebal,
// job 'S', reference LAPACK 3.5+ norms): for each index i, scale row i by 1/f and
// column i by f when that reduces ||col i||_2 + ||row i||_2 below 0.95 of its value;
// sweeps repeat until no index changes (at most 64 sweeps). scale[i] receives the
// accumulated factor; eigenvectors of the original matrix are diag(scale) times those
// of the balanced one. One workgroup per matrix.
__global__ __launch_bounds__(256) void balance_kernel(int N, cd* A, long lda, long sA, cd* scale, long ss) {
  __shared__ double red[4][4];
  __shared__ int changed;
  const long b = blockIdx.x;
  A += b * sA;
  scale += b * ss;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const double sfmin1 = SAFMIN / (ULP * 2.0), sfmax1 = 1.0 / sfmin1;
  const double sfmin2 = sfmin1 * 2.0, sfmax2 = 1.0 / sfmin2;
  for (int i = t; i < N; i += 256) scale[i] = mk(1.0, 0.0);
  __syncthreads();
  for (int sweep = 0; sweep < 64; ++sweep) {
    if (t == 0) changed = 0;
    __syncthreads();
    for (int i = 0; i < N; ++i) {
      // column and row 2-norms (with the diagonal) and largest moduli
      double c2 = 0.0, r2 = 0.0, ca = 0.0, ra = 0.0;
      for (int k = t; k < N; k += 256) {
        const cd cv = A[k + (long)i * lda], rv = A[i + (long)k * lda];
        c2 += cnorm2(cv);
        r2 += cnorm2(rv);
        ca = fmax(ca, cnorm2(cv));
        ra = fmax(ra, cnorm2(rv));
      }
      c2 = wsum(c2);
      r2 = wsum(r2);
      for (int o = 32; o > 0; o >>= 1) {
        ca = fmax(ca, __shfl_xor(ca, o, 64));
        ra = fmax(ra, __shfl_xor(ra, o, 64));
      }
      if (lane == 0) {
        red[0][wave] = c2;
        red[1][wave] = r2;
        red[2][wave] = ca;
        red[3][wave] = ra;
      }
      __syncthreads();
      double c = sqrt(red[0][0] + red[0][1] + red[0][2] + red[0][3]);
      double r = sqrt(red[1][0] + red[1][1] + red[1][2] + red[1][3]);
      ca = sqrt(fmax(fmax(red[2][0], red[2][1]), fmax(red[2][2], red[2][3])));
      ra = sqrt(fmax(fmax(red[3][0], red[3][1]), fmax(red[3][2], red[3][3])));
      __syncthreads();
      if (c == 0.0 || r == 0.0) continue;
      double g = r / 2.0, f = 1.0;
      const double s = c + r;
      while (c < g && fmax(f, fmax(c, ca)) < sfmax2 && fmin(r, fmin(g, ra)) > sfmin2) {
        f *= 2.0;
        c *= 2.0;
        ca *= 2.0;
        r /= 2.0;
        g /= 2.0;
        ra /= 2.0;
      }
      g = c / 2.0;
      while (g >= r && fmax(r, ra) < sfmax2 && fmin(fmin(f, c), fmin(g, ca)) > sfmin2) {
        f /= 2.0;
        c /= 2.0;
        g /= 2.0;
        ca /= 2.0;
        r *= 2.0;
        ra *= 2.0;
      }
      if (c + r >= 0.95 * s) continue;
      const double sc = scale[i].x;
      if (f < 1.0 && sc < 1.0 && f * sc <= sfmin1) continue;
      if (f > 1.0 && sc > 1.0 && sc >= sfmax1 / f) continue;
      const double gi = 1.0 / f;
      for (int k = t; k < N; k += 256) {
        A[i + (long)k * lda] = cscale(A[i + (long)k * lda], gi);
      }
      __syncthreads();
      for (int k = t; k < N; k += 256) {
        A[k + (long)i * lda] = cscale(A[k + (long)i * lda], f);
      }
      if (t == 0) {
        scale[i] = mk(sc * f, 0.0);
        changed = 1;
      }
      __syncthreads();
    }
    __syncthreads();
    if (!changed) break;
    __syncthreads();
  }
}

static int g_aed_window = -1;  // -1: automatic (aed_window_for)
static int g_bulges = 12;
static int g_max_sweeps = 0;  // 0: 30 * max(N, 10), LAPACK zlahqr's iteration budget
void zgeev_set_max_sweeps(int n) { g_max_sweeps = n < 0 ? 0 : n; }
void zgeev_set_aed(int window) { g_aed_window = window < -1 ? 0 : (window > QW ? QW : window); }
void zgeev_set_bulges(int nb) { g_bulges = nb < 1 ? 1 : (nb > NBUL ? NBUL : nb); }
// 0: hqr_kernel (W = 64, window products from registers), 1: hqr_lds_kernel (W = 64,
// window products staged through LDS), 2: hqr_w48_kernel (W = 48, two matrices per CU),
// 4: hqr_w32_kernel (W = 32, four matrices per CU); -1: automatic, 4 for N <= 256 in launches
// of at least 384 matrices and for N <= 512 in launches of at least 768, 2 for N <= 1024 in
// launches of at least 384, else 0. The lines are those of earlier kernels; with the present ones
// (QR stage of random matrices, ms, variants 0 / 2 / 4): N = 98 128 matrices 6.7 / 10.0 / 8.5, 384
// 13.3 / 12.1 / 10.8, 640 20.0 / 20.4 / 11.0; N = 162 384 29.1 / 24.1 / 28.5, 640 43.4 / 40.9 / 31.1;
// N = 242 384 54.4 / 46.4 / 67.4, 640 81.8 / 77.4 / 70.5, 1024 111 / 92 / 77; N = 338 384 101 / 86 / 150, 768
// 154 / 143 / 165; N = 450 384 174 / 158 / 313; N = 882 512 800 / 833. So variant 4 is early at N = 242 and 338,
// variant 2 late from N = 162 to 450 and, on these matrices, early at N = 882.
static int g_qr_variant = -1;
static int qr_variant_for(int n, int batch) {
  if (g_qr_variant >= 0) return g_qr_variant;
  if ((n <= 256 && batch >= 384) || (n <= 512 && batch >= 768)) return 4;
  if (n > 512 && n <= 1024 && batch >= 384) return 2;
  return 0;
}
static int g_bulges_w48 = 8;  // bulges per sweep of the W = 48 kernel (<= 12: >= 11 chase steps per window)
static int g_bulges_w32 = 6;  // bulges per sweep of the W = 32 kernel (<= 7: >= 10 chase steps per window)
void zgeev_set_qr_variant(int v) { g_qr_variant = (v < -1 || v > 4 || v == 3) ? -1 : v; }
void zgeev_set_bulges_w48(int nb) { g_bulges_w48 = nb < 1 ? 1 : (nb > 12 ? 12 : nb); }
void zgeev_set_bulges_w32(int nb) { g_bulges_w32 = nb < 1 ? 1 : (nb > 7 ? 7 : nb); }
int zgeev_get_bulges_w48() { return g_bulges_w48; }
int zgeev_get_bulges_w32() { return g_bulges_w32; }
int zgeev_get_qr_variant() { return g_qr_variant; }
// bit v set: QR kernel variant v was launched since the last zgeev_take_qr_kernels()
static std::atomic<unsigned> g_qr_ran{0};
unsigned zgeev_take_qr_kernels() { return g_qr_ran.exchange(0u); }
// QR workgroup slots of the GPU (256 CUs) for a variant: matrices one round of its
// workgroups holds
static int qr_slots(int v) { return v == 4 ? 1024 : (v == 2 ? 512 : 256); }
int zgeev_full_launch(int n) {
  return qr_slots(g_qr_variant >= 0 ? g_qr_variant : (n <= 512 ? 4 : (n <= 1024 ? 2 : 0)));
}
std::vector<int> zgeev_launch_plan(int n, int units, int per_unit) {
  std::vector<int> plan;
  if (units <= 0) return plan;
  if (per_unit < 1) per_unit = 1;
  const int full = zgeev_full_launch(n);
  const int per = full / per_unit > 1 ? full / per_unit : 1;
  plan.assign(units / per, per);
  if (units % per) plan.push_back(units % per);
  return plan;
}
// Deflation window of QR kernel variant v at size n. The window's Schur form is the longest
// serial part of a small problem, its deflations and shifts pay at large n. Measured best of
// 6 .. 28 (QR stage, ms; in brackets the former fixed 24): 64-wide kernel N = 50 8: 2.1 (5.3),
// N = 98 8: 6.3 (9.8), N = 126 12: 8.6, 8: 8.9, N = 162 16: 12.9, 12: 13.4, N = 242 16: 23.2
// (25.3), N = 338 16 and 24: 42.5, N = 450 24: 75.5, 16: 81.9, N = 882 24: 305, 20: 319; 32-wide
// kernel in full launches N = 98 8: 10.9 (17.6), N = 162 12: 27.7, 8: 29.3, N = 242 12: 61.1
// (74.2), N = 450 12 and 16: 296; 48-wide kernel N = 882 20: 688, 24: 691.
static int aed_window_for(int v, int n) {
  if (g_aed_window >= 0) return g_aed_window;
  if (v == 4) return n <= 128 ? 8 : 12;
  if (v == 2) return 20;
  return n <= 112 ? 8 : (n <= 144 ? 12 : (n <= 360 ? 16 : 24));
}
int zgeev_get_aed() { return g_aed_window; }
// Workgroups per matrix of the 64-wide kernel: what 32 CUs per XCD hold, at most 16. A member keeps
// its CU for the whole iteration, also while its master chases alone, so contexts on several streams
// of the process share the CUs out (up to four ways: HIP's hardware queues per process, by
// default); one launch holding all of them would make the others wait. Four contexts, ms a round
// with all CUs for each / a quarter / before there were teams: a stack of 10 layers each at N = 882
// 689 / 345 / 626, four at N = 450 300 / 181 / 227; a single matrix each at N = 882 179 / 193 / 483.
// The bits do not depend on the team. QR stage without / with a team below the line, ms: 8 matrices
// of N = 98 6.55 / 6.61, 126 9.76 / 9.82, 162 14.1 / 14.0, 198 19.2 / 18.3; 128 of N = 162 14.8 / 15.2.
static int team_size(int n, int batch, int streams) {
  if (n < 200 || n > 65535) return 1;
  const int per_xcd = (batch + 7) / 8;
  const int g = 32 / std::min(streams, 4) / per_xcd;
  return g < 16 ? g : 16;
}
int zgeev_get_bulges() { return g_bulges; }

// Schur factors of a strided batch (A destroyed): A = D Z T Z^H D^{-1} with D = diag(dbal)
// (balancing), Z unitary (ld n), T upper triangular (left in A); X (ld n, unit upper
// triangular) holds the eigenvectors of T, so that W = D Z X are eigenvectors of A
// (not normalized).
void zgeev_factors(hipStream_t s, int n, cd* A, long lda, long sA, cd* w, long sw, cd* Z, cd* X, cd* dbal,
                   int* info, int batch, Workspace& ws) {
  if (n <= 0 || batch <= 0) return;
  const long nn = (long)n * n;
  const int nref = n_reflectors(n);
  const int npanel = nref > 0 ? cdiv_up(nref, HB) : 1;
  DevBuf Tb = ws.get(sizeof(cd) * (size_t)npanel * HB * HB * batch);
  cd* Vf = X;  // the reflectors live in X until the eigenvectors overwrite them
  {
    StageScope st(ST_HESS);
    balance_kernel<<<batch, 256, 0, s>>>(n, A, lda, sA, dbal, n);
    launch_check("balance");
    gehrd(s, n, A, lda, sA, Vf, Tb.as<cd>(), batch, ws);
    orghr(s, n, Vf, Tb.as<cd>(), Z, n, nn, batch, ws);
  }
  {
    StageScope st(ST_QR);
    vrc_ctx* c = tl_ctx();
    const bool want = c && c->timing;
    DevBuf sb;
    if (want) sb = ws.get(sizeof(long long) * 5 * batch);
    long long* stp = want ? sb.as<long long>() : nullptr;
    const int qv = qr_variant_for(n, batch);
    g_qr_ran.fetch_or(1u << qv, std::memory_order_relaxed);
    const int aed = aed_window_for(qv, n);
    if (qv == 4) {
      hqr_w32_kernel<<<batch, 128, 0, s>>>(n, A, lda, sA, Z, n, nn, w, sw, info, stp, aed, g_bulges_w32,
                                           g_max_sweeps);
    } else if (qv == 2) {
      hqr_w48_kernel<<<batch, 256, 0, s>>>(n, A, lda, sA, Z, n, nn, w, sw, info, stp, aed, g_bulges_w48,
                                           g_max_sweeps);
    } else if (qv == 1) {
      hqr_lds_kernel<<<batch, QT, 0, s>>>(n, A, lda, sA, Z, n, nn, w, sw, info, stp, aed, g_bulges,
                                          g_max_sweeps);
    } else if (const int team = team_size(n, batch, gpu_streams(c ? c->device : 0)); team > 1) {
      const int batch8 = (batch + 7) & ~7;
      DevBuf tc = ws.get(sizeof(TeamCtl) * (size_t)batch), tu = ws.get(sizeof(cd) * (size_t)QW * QW * batch);
      fill_int(s, tc.as<int>(), 0, (int)(sizeof(TeamCtl) / sizeof(int)) * batch);
      hqr_team_kernel<<<batch8 * team, QT, 0, s>>>(n, A, lda, sA, Z, n, nn, w, sw, info, stp, aed, g_bulges,
                                                   g_max_sweeps, batch, batch8, tc.as<TeamCtl>(), tu.as<cd>());
    } else {
      hqr_kernel<<<batch, QT, 0, s>>>(n, A, lda, sA, Z, n, nn, w, sw, info, stp, aed, g_bulges,
                                      g_max_sweeps);
    }
    launch_check("hqr");
    health_note_info(s, info, batch, H_EIG);
    if (want) {
      std::vector<long long> h(5 * (size_t)batch);
      VRC_HIP(hipMemcpyAsync(h.data(), sb.ptr, sizeof(long long) * h.size(), hipMemcpyDeviceToHost, s));
      VRC_HIP(hipStreamSynchronize(s));
      c->qr_stats[0] += batch;
      for (int b = 0; b < batch; ++b)
        for (int k = 0; k < 5; ++k) c->qr_stats[1 + k] += h[(size_t)b * 5 + k];
    }
  }
  StageScope st(ST_EIGVEC);
  zset(s, n, n, mk(0.0, 0.0), mk(0.0, 0.0), X, n, nn, batch);
  dim3 g(cdiv_up(n, QW), batch);
  trevc_kernel<<<g, 256, 0, s>>>(n, A, lda, sA, X, n, nn);
  launch_check("trevc");
}

// VR = D Z X with LAPACK zgeev's normalisation (unit 2-norm, largest component real).
void zgeev_vectors(hipStream_t s, int n, const cd* Z, const cd* X, const cd* dbal, cd* VR, long ldv, long sV,
                   int batch) {
  if (n <= 0 || batch <= 0) return;
  StageScope st(ST_EIGVEC);
  const long nn = (long)n * n;
  zgemm_strided(s, OP_N, OP_N, n, n, n, mk(1.0, 0.0), Z, n, nn, X, n, nn, mk(0.0, 0.0), VR, ldv, sV, batch);
  zdscale(s, n, n, dbal, n, nullptr, 0, 0, VR, ldv, sV, VR, ldv, sV, batch);  // undo the balancing
  dim3 gn(cdiv_up(n, 4), batch);
  normalize_cols_kernel<<<gn, 256, 0, s>>>(n, VR, ldv, sV);
  launch_check("normalize_cols");
}

void zgeev_batched(hipStream_t s, int n, cd* A, long lda, long sA, cd* w, long sw, cd* VR, long ldv, long sV,
                   int* info, int batch, Workspace& ws) {
  if (n <= 0 || batch <= 0) return;
  const long nn = (long)n * n;
  DevBuf Zb = ws.get(sizeof(cd) * (size_t)nn * batch), Xb = ws.get(sizeof(cd) * (size_t)nn * batch);
  DevBuf Db = ws.get(sizeof(cd) * (size_t)n * batch);
  zgeev_factors(s, n, A, lda, sA, w, sw, Zb.as<cd>(), Xb.as<cd>(), Db.as<cd>(), info, batch, ws);
  zgeev_vectors(s, n, Zb.as<cd>(), Xb.as<cd>(), Db.as<cd>(), VR, ldv, sV, batch);
}

__global__ void gamma_sqrt_kernel(int n, const cd* lam, long sl, cd* gam, long sg) {
  const long b = blockIdx.y;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  gam[b * sg + i] = gamma_branch(lam[b * sl + i]);
}

void gamma_sqrt(hipStream_t s, int n, const cd* lam, long sl, cd* gam, long sg, int batch) {
  if (n <= 0 || batch <= 0) return;
  dim3 g(cdiv_up(n, 256), batch);
  gamma_sqrt_kernel<<<g, 256, 0, s>>>(n, lam, sl, gam, sg);
  launch_check("gamma_sqrt");
  if (sg == n) health_note_gamma(s, gam, (long)n * batch);
}

}  // namespace vrc
