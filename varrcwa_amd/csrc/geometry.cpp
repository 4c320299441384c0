// Host-side geometry preparation: painter-order refill, K matrices (periodic and
// PML-stretched), and upload of a layer batch for the Fourier assembly kernels.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>

#include "vrc_ops.hpp"

namespace vrc {

static constexpr double PI_REF = 3.1415926535897932;  // src/rcwa/defns.h:29

static double sinc_ref(double x) { return x == 0.0 ? 1.0 : std::sin(PI_REF * x) / (PI_REF * x); }
static cd cexp_i(double a) { return mk(std::cos(a), std::sin(a)); }
static cd hmul(cd a, cd b) { return cmul(a, b); }

static void bad_permittivity(const double* e, size_t n) {
  for (size_t i = 0; i < n; ++i) {
    if (!std::isfinite(e[2 * i]) || !std::isfinite(e[2 * i + 1]))
      throw ArgFailure("non-finite permittivity (NaN or infinity)");
    // the inverse Fourier rules (fe11, fe22) are built from 1/eps of every cell
    if (e[2 * i] == 0.0 && e[2 * i + 1] == 0.0)
      throw ArgFailure("zero permittivity in a cell: the inverse Fourier rules need 1/eps");
  }
}

// Checks a layer's permittivities and, with out, copies them, in one pass.
template <bool COPY>
static void scan_permittivity(const LayerView& L, double* out) {
  const double* e = L.eps;
  const size_t n = L.neps;
  double nf[4] = {0.0, 0.0, 0.0, 0.0};  // NaN once a value is not finite; four independent sums
  bool zero = false;
  size_t i = 0;
  for (; i + 2 <= n; i += 2) {
    const double* q = e + 2 * i;
    for (int r = 0; r < 4; ++r) nf[r] += q[r] * 0.0;
    zero |= ((q[0] == 0.0) & (q[1] == 0.0)) | ((q[2] == 0.0) & (q[3] == 0.0));
    if (COPY)
      for (int r = 0; r < 4; ++r) out[2 * i + r] = q[r];
  }
  if (i < n) {
    nf[0] += e[2 * i] * 0.0 + e[2 * i + 1] * 0.0;
    zero |= (e[2 * i] == 0.0) & (e[2 * i + 1] == 0.0);
    if (COPY) {
      out[2 * i] = e[2 * i];
      out[2 * i + 1] = e[2 * i + 1];
    }
  }
  if (zero || !(nf[0] + nf[1] + nf[2] + nf[3] == 0.0)) bad_permittivity(e, n);
}

PreparedLayer prepare_layer(const LayerView& L) {
  const int nCx = L.ncoord_x, nCy = L.ncoord_y;
  if (nCx < 2 || nCy < 2) throw ArgFailure("layer needs at least 2 coordinates per axis");
  if (L.neps != (size_t)(nCx - 1) * (nCy - 1)) throw ArgFailure("eps size does not match coordinates");
  PreparedLayer p;
  p.ncx = nCx - 1;
  p.ncy = nCy - 1;
  p.Lx = L.x[nCx - 1] - L.x[0];
  p.Ly = L.y[nCy - 1] - L.y[0];
  p.xu.assign(L.x, L.x + nCx);
  p.ys.assign(L.y, L.y + nCy);
  // FourierSolver1D::reorder: indices sorted by coordinate (stable for ties)
  std::vector<int> index(nCx), rindex(nCx);
  std::iota(index.begin(), index.end(), 0);
  std::stable_sort(index.begin(), index.end(), [&](int a, int b) { return L.x[a] < L.x[b]; });
  for (int i = 0; i < nCx; ++i) rindex[index[i]] = i;
  p.xs.resize(nCx);
  for (int i = 0; i < nCx; ++i) p.xs[i] = L.x[index[i]];
  bool refill = false;
  for (int i = 0; i + 1 < nCx; ++i)
    if (rindex[i] != i) { refill = true; break; }
  p.src.resize(p.ncx);
  std::iota(p.src.begin(), p.src.end(), 0);
  // painter's order: cell i covers sorted intervals rindex[i] .. rindex[i+1]-1
  for (int i = 0; refill && i < p.ncx; ++i) {
    if (L.x[i] >= L.x[i + 1]) continue;
    for (int j = 0; j < p.ncx; ++j)
      if (rindex[i] <= j && rindex[i + 1] >= j + 1) p.src[j] = i;
  }
  return p;
}

void validate_layer(const HostLayer& L) {
  prepare_layer(L);
  scan_permittivity<false>(L, nullptr);
}

void alpha_beta(int nx, int ny, double Lx, double Ly, std::vector<cd>& alpha, std::vector<cd>& beta) {
  const int Nx = (nx - 1) / 2, Ny = (ny - 1) / 2;
  const double Kx = 2 * PI_REF / Lx, Ky = 2 * PI_REF / Ly;
  alpha.assign((size_t)nx * ny, mk(0, 0));
  beta.assign((size_t)nx * ny, mk(0, 0));
  for (int i = 0; i < nx; ++i)
    for (int j = 0; j < ny; ++j) {
      alpha[(size_t)ny * i + j] = mk(Kx * (double)(i - Nx), 0.0);
      beta[(size_t)ny * i + j] = mk(Ky * (double)(j - Ny), 0.0);
    }
}

// PMLSolver1D::solve (src/rcwa/PMLSolver1D.cpp:15-30)
static cd pml1d(double b0, double b1, double L, cd gamma, int n, double coeff) {
  const double bm = (b1 - b0) / L, bp = (b1 + b0) / L;
  auto ex = [](double x) { return cexp_i(PI_REF * x); };
  cd r = cscale(ex(-(n * bp + coeff * 0.5)), 4.0 * sinc_ref(n * bm - 0.5));
  r = cadd(r, cscale(ex(-(n * bp)), 8.0 * sinc_ref(n * bm)));
  r = cadd(r, cscale(hmul(gamma, ex(-(n * bp))), -2.0 * sinc_ref(n * bm)));
  r = cadd(r, cscale(ex(-(n * bp - coeff * 0.5)), 4.0 * sinc_ref(n * bm + 0.5)));
  r = cadd(r, cscale(hmul(gamma, ex(-(n * bp + coeff * 1.0))), sinc_ref(n * bm - 1.0)));
  r = cadd(r, cscale(hmul(gamma, ex(-(n * bp - coeff * 1.0))), sinc_ref(n * bm + 1.0)));
  return cscale(r, bm / 16.0);
}

// VarLayerSampler::assignSimulationRegion (src/core/VarLayerSampler.cpp:23-39): the cell
// and the absorbing regions from the first/last two coordinates of each axis.
Region region_from_coords(const std::vector<double>& x, const std::vector<double>& y) {
  const int nCx = (int)x.size(), nCy = (int)y.size();
  Region r;
  r.Lx = x[nCx - 1] - x[0];
  r.Ly = y[nCy - 1] - y[0];
  r.b0 = y[0];
  r.b1 = nCy > 1 ? y[1] : y[0];
  r.u0 = nCy > 1 ? y[nCy - 2] : y[0];
  r.u1 = y[nCy - 1];
  r.l0 = x[0];
  r.l1 = nCx > 1 ? x[1] : x[0];
  r.r0 = nCx > 1 ? x[nCx - 2] : x[0];
  r.r1 = x[nCx - 1];
  return r;
}

void pml_k_matrices(int nx, int ny, const std::vector<double>& x, const std::vector<double>& y,
                    std::vector<cd>& Kx, std::vector<cd>& Ky) {
  pml_k_matrices(nx, ny, region_from_coords(x, y), Kx, Ky);
}

// LayerSampler::evaluateKMatrices + evaluatePML (src/core/LayerSampler.cpp:34-132) for a
// region given by its scalars.
void pml_k_matrices(int nx, int ny, const Region& R, std::vector<cd>& Kx, std::vector<cd>& Ky) {
  const double Lx = R.Lx, Ly = R.Ly;
  const double b0 = R.b0, b1 = R.b1, u0 = R.u0, u1 = R.u1;
  const double l0 = R.l0, l1 = R.l1, r0 = R.r0, r1 = R.r1;
  std::vector<cd> alpha, beta;
  alpha_beta(nx, ny, Lx, Ly, alpha, beta);
  const cd gamma = crecip(mk(1.0, -1.0));
  const int nPx = 2 * nx - 1, nPy = 2 * ny - 1, maxPx = (nPx - 1) / 2, maxPy = (nPy - 1) / 2;
  std::vector<cd> fyy(nPy), fxx(nPx), fyx(nPx), fxy(nPy);
  for (int i = 0; i < nPy; ++i) {
    const int n = i - maxPy;
    cd v = cdiv(mk((u0 - b1) / Ly * sinc_ref(n * (u0 - b1) / Ly), 0.0), cexp_i(PI_REF * (n * (b1 + u0) / Ly)));
    v = cadd(v, pml1d(b0, b1, Ly, gamma, n, 1.0));
    fyy[i] = cadd(v, pml1d(u0, u1, Ly, gamma, n, -1.0));
  }
  for (int i = 0; i < nPx; ++i) {
    const int m = i - maxPx;
    cd v = cdiv(mk((r0 - l1) * sinc_ref(m * (r0 - l1) / Lx) / Lx, 0.0), cexp_i(PI_REF * m * (l1 + r0) / Lx));
    v = cadd(v, pml1d(l0, l1, Lx, gamma, m, 1.0));
    fxx[i] = cadd(v, pml1d(r0, r1, Lx, gamma, m, -1.0));
  }
  for (int i = 0; i < nPx; ++i) {
    const int m = i - maxPx;
    fyx[i] = (m == 0) ? mk(r1 - l0, 0.0)
                      : cmul(csub(cexp_i(-2 * PI_REF / Lx * m * r1), cexp_i(-2 * PI_REF / Lx * m * l0)),
                             mk(0.0, Lx * Lx / (m * 2 * PI_REF)));
  }
  for (int i = 0; i < nPy; ++i) {
    const int n = i - maxPy;
    fxy[i] = (n == 0) ? mk(u1 - b0, 0.0)
                      : cmul(csub(cexp_i(-2 * PI_REF / Ly * n * u1), cexp_i(-2 * PI_REF / Ly * n * b0)),
                             mk(0.0, Ly * Ly / (2 * n * PI_REF)));
  }
  // fy = fyx fyy^T / Lx ; fx = fxx fxy^T / Ly ; K = BlockToeplitz(f) * diag(alpha/beta)
  const int n = nx * ny;
  Kx.assign((size_t)n * n, mk(0, 0));
  Ky.assign((size_t)n * n, mk(0, 0));
  for (int r = 0; r < n; ++r)
    for (int c = 0; c < n; ++c) {
      const int m = r / ny, nn = r % ny, j = c / ny, l = c % ny;
      const int p = nx - 1 + (m - j), q = ny - 1 + (nn - l);
      const cd fx = cscale(cmul(fxx[p], fxy[q]), 1.0 / Ly);
      const cd fy = cscale(cmul(fyx[p], fyy[q]), 1.0 / Lx);
      Kx[(size_t)r + (size_t)c * n] = cmul(fx, alpha[c]);
      Ky[(size_t)r + (size_t)c * n] = cmul(fy, beta[c]);
    }
}

__global__ void fill_int_kernel(int* p, int v, long n) {
  long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

void fill_int(hipStream_t s, int* p, int v, long n) {
  if (n <= 0) return;
  fill_int_kernel<<<cdiv_up(n, 256), 256, 0, s>>>(p, v, n);
  launch_check("fill_int");
}

// val[l][strip][cell] from the layers' values as given (raw: one layer after the other from
// off[l], ncy x ncx column-major) through the painter's order src; cells past a layer's own are 1.
// A 16 x 16 tile goes through LDS so that both sides are read and written along their rows.
__global__ __launch_bounds__(256) void order_cells_kernel(const cd* raw, const long* off, const int* src,
                                                          const int* ncx, const int* ncy, int MX, int MY, cd* val) {
  __shared__ cd tile[16][17];
  const int l = blockIdx.z, cx = ncx[l], cy = ncy[l];
  const int j0 = blockIdx.x * 16, s0 = blockIdx.y * 16;
  const int a = threadIdx.x & 15, b = threadIdx.x >> 4;
  const bool in = j0 + b < cx && s0 + a < cy;
  tile[b][a] = in ? raw[off[l] + (s0 + a) + (long)src[(long)l * MX + j0 + b] * cy] : mk(1.0, 0.0);
  __syncthreads();
  if (j0 + a < MX && s0 + b < MY) val[((long)l * MY + s0 + b) * MX + j0 + a] = tile[a][b];
}

// Does the host write the cells in painter's order? Up to these counts (padded) the strided write
// costs less than order_cells_kernel (us, host / kernel, 3 x 3 harmonics): 1 layer of 1 cell 42 / 62, 64
// of 8 x 8 124 / 149, 2 of 20 x 20 69 / 80, 3 of 50 x 50 130 / 136, 8 of 32 x 32 100 / 105;
// 16 of 32 x 32 124 / 121, 1 of 64 x 64 90 / 84, 2 of 64 x 64 104 / 88, 2 of 128 x 128 239 / 123.
static bool host_orders_cells(size_t per_layer, int layers) { return per_layer < 4096 && per_layer * layers <= 12288; }

FourierStage fourier_prepare(vrc_ctx& c, int nx, int ny, const std::vector<const HostLayer*>& layers) {
  std::vector<LayerView> v;
  v.reserve(layers.size());
  for (const HostLayer* l : layers) v.emplace_back(*l);
  return fourier_prepare(c, nx, ny, v);
}

FourierStage fourier_prepare(vrc_ctx& c, int nx, int ny, const std::vector<LayerView>& layers) {
  hipStream_t s = c.stream;
  const int L = (int)layers.size();
  FourierStage fs;
  fs.L = L;
  std::vector<PreparedLayer> pl;
  pl.reserve(L);
  int MX = 1, MY = 1;
  std::vector<long> off(L);
  long cells = 0;
  for (int l = 0; l < L; ++l) {
    pl.push_back(prepare_layer(layers[l]));
    MX = std::max(MX, pl.back().ncx);
    MY = std::max(MY, pl.back().ncy);
    off[l] = cells;
    cells += (long)layers[l].neps;
  }
  const int M1 = 2 * nx - 1, M2 = 2 * ny - 1;
  // uniform power-of-two grids along x (sorted, so no refill) and y take the FFT path
  auto fft_log2 = [](const std::vector<double>& c, const std::vector<double>* sorted) -> int {
    const int n = (int)c.size() - 1;
    if (n < 2 || n > FOURIER_FFT_MAX || (n & (n - 1)) != 0) return 0;
    if (sorted && *sorted != c) return 0;
    const double d = c[n] - c[0];
    if (!(d > 0)) return 0;
    for (int j = 0; j <= n; ++j)
      if (std::fabs(c[j] - (c[0] + d * j / n)) > 1e-12 * d) return 0;
    int lg = 0;
    while ((1 << lg) < n) ++lg;
    return lg;
  };
  std::vector<int> fx(L), fy(L);
  int fft_max = 0;
  for (int l = 0; l < L; ++l) {
    fx[l] = fft_log2(pl[l].xu, &pl[l].xs);
    fy[l] = fft_log2(pl[l].ys, nullptr);
    fft_max = std::max(fft_max, std::max(fx[l] ? 1 << fx[l] : 0, fy[l] ? 1 << fy[l] : 0));
  }
  // One upload: the geometry, then the layers' values as they were given, checked and written
  // straight into the pinned block; the device (for few cells the host, host_orders_cells) puts
  // the cells into painter's order. 64 layers of 256 x 256 cells, assembled: 3.3 ms, of which 1.3
  // are the copy to the device; through six host arrays and a strided transpose it took 56.
  const size_t od = sizeof(int) * 4 * L, ox = od + sizeof(double) * 2 * L,
               oy = ox + sizeof(double) * 2 * (size_t)L * (MX + 1), oo = oy + sizeof(double) * (size_t)L * (MY + 1),
               os = oo + sizeof(long) * L, geo_bytes = (os + sizeof(int) * (size_t)L * MX + 15) & ~(size_t)15;
  const size_t nval = (size_t)MY * MX;
  const bool host_order = host_orders_cells(nval, L);
  const size_t val_bytes = sizeof(cd) * (host_order ? nval * L : (size_t)cells);
  fs.geo = c.ws.get(geo_bytes + val_bytes);
  c.pinned.upload_with(s, fs.geo.ptr, geo_bytes + val_bytes, [&](char* h) {
    std::memset(h, 0, geo_bytes);
    int* hi = (int*)h;
    double *hd = (double*)(h + od), *hx = (double*)(h + ox), *hy = (double*)(h + oy);
    long* ho = (long*)(h + oo);
    int* hs = (int*)(h + os);
    for (int l = 0; l < L; ++l) {
      const PreparedLayer& p = pl[l];
      hi[l] = p.ncx;
      hi[L + l] = p.ncy;
      hi[2 * L + l] = fx[l];
      hi[3 * L + l] = fy[l];
      hd[l] = p.Lx;
      hd[L + l] = p.Ly;
      std::copy(p.xu.begin(), p.xu.end(), hx + (size_t)l * (MX + 1));
      std::copy(p.xs.begin(), p.xs.end(), hx + (size_t)(L + l) * (MX + 1));
      std::copy(p.ys.begin(), p.ys.end(), hy + (size_t)l * (MY + 1));
      ho[l] = off[l];
      std::copy(p.src.begin(), p.src.end(), hs + (size_t)l * MX);
    }
    double* hv = (double*)(h + geo_bytes);
    if (!host_order) {
      for (int l = 0; l < L; ++l) scan_permittivity<true>(layers[l], hv + 2 * off[l]);
      return;
    }
    cd* v = (cd*)hv;
    std::fill(v, v + nval * L, mk(1.0, 0.0));
    for (int l = 0; l < L; ++l, v += nval) {
      const PreparedLayer& p = pl[l];
      scan_permittivity<false>(layers[l], nullptr);
      for (int j = 0; j < p.ncx; ++j) {
        const double* e = layers[l].eps + 2 * (size_t)p.src[j] * p.ncy;  // 8-byte aligned only
        for (int i = 0; i < p.ncy; ++i) v[(size_t)i * MX + j] = mk(e[2 * i], e[2 * i + 1]);
      }
    }
  });
  char* d = (char*)fs.geo.ptr;
  FourierDev& g = fs.g;
  g.nx = nx;
  g.ny = ny;
  g.MX = MX;
  g.MY = MY;
  g.ncx = (const int*)d;
  g.ncy = (const int*)d + L;
  g.fftx = (const int*)d + 2 * L;
  g.ffty = (const int*)d + 3 * L;
  g.fft_max = fft_max;
  const double* dd = (const double*)(d + od);
  g.Lx = dd;
  g.Ly = dd + L;
  g.xu = dd + 2 * L;
  g.xs = g.xu + (size_t)L * (MX + 1);
  g.ys = g.xs + (size_t)L * (MX + 1);
  const size_t nFX = (size_t)MY * M1, nFY1 = (size_t)MY * M2, nFYi = (size_t)MX * M2, nFX1 = (size_t)MX * M1,
               ntx = (size_t)MY * nx * nx, nty = (size_t)MX * ny * ny, nF2 = (size_t)M1 * M2,
               nG11 = (size_t)nx * nx * M2, nG22 = (size_t)ny * ny * M1;
  const size_t per = 2 * nFX + nFY1 + nFYi + nFX1 + ntx + nty + nF2 + nG11 + nG22;
  fs.wk = c.ws.get(sizeof(cd) * (per + (host_order ? 0 : nval)) * L);
  cd* w = fs.wk.as<cd>();
  if (host_order) {
    g.val = (const cd*)(d + geo_bytes);
  } else {
    order_cells_kernel<<<dim3(cdiv_up(MX, 16), cdiv_up(MY, 16), L), 256, 0, s>>>(
        (const cd*)(d + geo_bytes), (const long*)(d + oo), (const int*)(d + os), g.ncx, g.ncy, MX, MY, w);
    launch_check("order_cells");
    g.val = w;
    w += nval * L;
  }
  g.FX = w;
  g.FXi = g.FX + nFX * L;
  g.FY1 = g.FXi + nFX * L;
  g.FYi = g.FY1 + nFY1 * L;
  g.FX1 = g.FYi + nFYi * L;
  g.tFFx = g.FX1 + nFX1 * L;
  g.tFFy = g.tFFx + ntx * L;
  g.F2 = g.tFFy + nty * L;
  g.G11 = g.F2 + nF2 * L;
  g.G22 = g.G11 + nG11 * L;
  return fs;
}

void assemble_fe(vrc_ctx& c, const AssemblyBatch& a, cd* fe11, cd* fe22, cd* fe33, long sfe) {
  std::vector<LayerView> v;
  v.reserve(a.layers.size());
  for (const HostLayer* l : a.layers) v.emplace_back(*l);
  assemble_fe(c, a.nx, a.ny, v, fe11, fe22, fe33, sfe);
}

void assemble_fe(vrc_ctx& c, int nx, int ny, const std::vector<LayerView>& layers, cd* fe11, cd* fe22, cd* fe33,
                 long sfe) {
  FourierStage fs = fourier_prepare(c, nx, ny, layers);
  StageScope st(ST_FOURIER);
  fourier_assemble(c.stream, fs.g, fs.L, fe11, fe22, fe33, sfe);
}

}  // namespace vrc
