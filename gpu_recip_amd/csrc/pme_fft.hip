// pme_fft.hip -- 3-D real-to-complex FFT of the PME grid and the reciprocal
// convolution (scalar sum), hand-written for CDNA4.
//
// Layouts (the reference's BOX layout, CudaPMERecip.cu:1383, 1399-1400):
//   real grid     float [nz][ny][nx]            (x fastest, packed)
//   half spectrum float2[nz][ny][nx/2+1]        (x fastest)
// Forward transforms use e^{-2 pi i}, inverse e^{+2 pi i}, both unnormalised.
//
// Passes: x (R2C / C2R over rows, even nx through a half-length complex FFT),
// y and z over strided columns, tiled as TX consecutive kx so every HBM access
// is a contiguous run.  Every 1-D transform runs in LDS as mixed-radix
// (2/3/4/5/8) Stockham stages.  The z pass can run forward FFT -> influence
// function (energy/virial in FP64) -> inverse FFT in one kernel, which is the
// reference's r2c z-stage + scalar_sum + c2r z-stage in one read and one write
// of the spectrum.
#include "pme_internal.hpp"
#include "pme_zpass.hpp"

namespace pme {

// ---------------------------------------------------------------- x pass ----

// Row tile `tile` (NR rows) of one grid; sm: dynamic LDS (fft_x_lds_bytes).
// Offset of spectrum row r (= ky + ny kz) in the padded half spectrum.
__device__ __forceinline__ size_t spec_row(int r, int ny, int hx, long long pz) {
  const int kz = sdiv(r, small_div(ny));
  return (size_t)kz * (size_t)pz + (size_t)(r - kz * ny) * hx;
}

__device__ __forceinline__ void fft_x_r2c_body(const float* __restrict__ grid, float2* __restrict__ cg, int nx,
                                               int nrows, int ny, int NR, const AxisArgs& ax, int tile, float2* sm) {
  const int tid = threadIdx.x;
  const int nf = ax.rp.n;
  const int LS = NR + 1;
  float2* tw = sm;
  float2* b0 = sm + ax.ntw;
  float2* b1 = b0 + nf * LS;
  for (int i = tid; i < ax.ntw; i += kBlock) tw[i] = ax.tw[i];
  const int row0 = tile * NR;
  const int nr = min(NR, nrows - row0);
  const int hx = nx / 2 + 1;
  const bool even = (nx & 1) == 0;
  if (even) {
    // the tile's rows are contiguous in HBM: keep U loads in flight per thread
    const float2* src = reinterpret_cast<const float2*>(grid + (size_t)row0 * nx);
    const int ntile = NR * nf, nvalid = nr * nf;
    for (int e0 = tid; e0 < ntile; e0 += kStageU * kBlock) {
      float2 v[kStageU];
#pragma unroll
      for (int u = 0; u < kStageU; u++) {
        const int e = e0 + u * kBlock;
        v[u] = (e < nvalid) ? src[e] : make_float2(0.f, 0.f);
      }
#pragma unroll
      for (int u = 0; u < kStageU; u++) {
        const int e = e0 + u * kBlock;
        if (e < ntile) {
          const int row = sdiv(e, small_div(nf));
          b0[(e - row * nf) * LS + row] = v[u];
        }
      }
    }
  } else {
    const float* src = grid + (size_t)row0 * nx;
    const int ntile = NR * nx, nvalid = nr * nx;
    for (int e0 = tid; e0 < ntile; e0 += kStageU * kBlock) {
      float v[kStageU];
#pragma unroll
      for (int u = 0; u < kStageU; u++) {
        const int e = e0 + u * kBlock;
        v[u] = (e < nvalid) ? src[e] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < kStageU; u++) {
        const int e = e0 + u * kBlock;
        if (e < ntile) {
          const int row = sdiv(e, small_div(nx));
          b0[(e - row * nx) * LS + row] = make_float2(v[u], 0.f);
        }
      }
    }
  }
  __syncthreads();
  float2* res = fft_lines<-1>(b0, b1, tw, ax.rp, NR, LS, tid, kBlock);
  if (even) {
    // X[k] = E[k] + w^k O[k], E = (Z[k] + Z*[h-k])/2, O = (Z[k] - Z*[h-k])/(2i)
    const int h = nf;
    for (int e = tid; e < nr * hx; e += kBlock) {
      const int row = sdiv(e, small_div(hx));
      const int k = e - row * hx;
      const float2 zk = res[(k == h ? 0 : k) * LS + row];
      const float2 zc = cconj(res[(k == 0 ? 0 : h - k) * LS + row]);
      const float2 E = cscale(cadd(zk, zc), 0.5f);
      const float2 D = csub(zk, zc);
      const float2 O = make_float2(0.5f * D.y, -0.5f * D.x);
      cg[spec_row(row0 + row, ny, hx, spec_pitch(hx, ny)) + k] = cadd(E, cmul(tw[k], O));
    }
  } else {
    for (int e = tid; e < nr * hx; e += kBlock) {
      const int row = sdiv(e, small_div(hx));
      const int k = e - row * hx;
      cg[spec_row(row0 + row, ny, hx, spec_pitch(hx, ny)) + k] = res[k * LS + row];
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_fft_x_r2c(const float* __restrict__ grid, float2* __restrict__ cg, int nx,
                                                      int nrows, int ny, int NR, AxisArgs ax) {
  extern __shared__ __align__(16) float2 sm[];
  fft_x_r2c_body(grid, cg, nx, nrows, ny, NR, ax, blockIdx.x, sm);
}

__device__ __forceinline__ void fft_x_c2r_body(const float2* __restrict__ cg, float* __restrict__ grid, int nx,
                                               int nrows, int ny, int NR, const AxisArgs& ax, int tile, float2* sm) {
  const int tid = threadIdx.x;
  const int nf = ax.rp.n;
  const int LS = NR + 1;
  float2* tw = sm;
  float2* b0 = sm + ax.ntw;
  float2* b1 = b0 + nf * LS;
  for (int i = tid; i < ax.ntw; i += kBlock) tw[i] = ax.tw[i];
  __syncthreads();
  const int row0 = tile * NR;
  const int nr = min(NR, nrows - row0);
  const int hx = nx / 2 + 1;
  const bool even = (nx & 1) == 0;
  if (even) {
    // Z[k] = (X[k] + X*[h-k]) + i w^{-k} (X[k] - X*[h-k]),  k < h
    const int h = nf;
    for (int e0 = tid; e0 < NR * h; e0 += kStageU * kBlock) {
      float2 xk[kStageU], xc[kStageU];
#pragma unroll
      for (int u = 0; u < kStageU; u++) {
        const int e = e0 + u * kBlock;
        const int row = sdiv(e, small_div(h));
        const int k = e - row * h;
        xk[u] = xc[u] = make_float2(0.f, 0.f);
        if (row < nr) {
          const float2* x = cg + spec_row(row0 + row, ny, hx, spec_pitch(hx, ny));
          xk[u] = x[k];
          xc[u] = cconj(x[h - k]);
        }
      }
#pragma unroll
      for (int u = 0; u < kStageU; u++) {
        const int e = e0 + u * kBlock;
        if (e < NR * h) {
          const int row = sdiv(e, small_div(h));
          const int k = e - row * h;
          const float2 A = cadd(xk[u], xc[u]);
          const float2 B = cmul(cconj(tw[k]), csub(xk[u], xc[u]));
          b0[k * LS + row] = make_float2(A.x - B.y, A.y + B.x);
        }
      }
    }
  } else {
    for (int e = tid; e < NR * nx; e += kBlock) {
      const int row = sdiv(e, small_div(nx));
      const int k = e - row * nx;
      float2 z = make_float2(0.f, 0.f);
      if (row < nr) {
        const float2* x = cg + spec_row(row0 + row, ny, hx, spec_pitch(hx, ny));
        z = (k < hx) ? x[k] : cconj(x[nx - k]);
      }
      b0[k * LS + row] = z;
    }
  }
  __syncthreads();
  float2* res = fft_lines<+1>(b0, b1, tw, ax.rp, NR, LS, tid, kBlock);
  if (even) {
    float2* dst = reinterpret_cast<float2*>(grid + (size_t)row0 * nx);
    for (int e = tid; e < nr * nf; e += kBlock) {
      const int row = sdiv(e, small_div(nf));
      const int m = e - row * nf;
      dst[(size_t)row * nf + m] = res[m * LS + row];
    }
  } else {
    for (int e = tid; e < nr * nx; e += kBlock) {
      const int row = sdiv(e, small_div(nx));
      const int m = e - row * nx;
      grid[(size_t)(row0 + row) * nx + m] = res[m * LS + row].x;
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_fft_x_c2r(const float2* __restrict__ cg, float* __restrict__ grid, int nx,
                                                      int nrows, int ny, int NR, AxisArgs ax) {
  extern __shared__ __align__(16) float2 sm[];
  fft_x_c2r_body(cg, grid, nx, nrows, ny, NR, ax, blockIdx.x, sm);
}

// ------------------------------------------------------------- xy planes --
// One workgroup transforms np (1 or 2) consecutive z planes through x and y
// in LDS, so each plane is read once and written once with contiguous
// accesses:
//   forward: real rows --x R2C--> half-spectrum rows, transposed in LDS to
//            columns --y FFT--> the planes of the half spectrum;
//   inverse: the reverse (y inverse, C2R pre-processing, x inverse).
// The rows of the np planes are one batch of np*ny x lines (row r of plane p
// is line p*ny + r, the order they have in memory), and their columns one
// batch of np*hx y lines (column k of plane p is line p*hx + k), so two
// planes share every FFT stage and barrier.
// LDS: twiddles of x and y, two buffers of plane_buf() points.  x lines
// have point stride LSX, y lines point stride LSY, both odd so that 8-byte
// accesses of consecutive lines hit distinct bank pairs.
// Odd nx: rows 2j and 2j+1 of a plane are the real and imaginary parts of
// one x line (one complex FFT of length nx transforms two rows; an odd ny
// pairs the plane's last row with zeros), so a plane has (ny + 1) / 2 x
// lines; the pairs never cross planes, so a group of planes rounds exactly
// as its planes one at a time.

__host__ __device__ constexpr int odd_pad(int n) { return (n + 1) | 1; }

// x lines of one plane
__host__ __device__ constexpr int plane_xlines(int nx, int ny) { return (nx & 1) ? (ny + 1) >> 1 : ny; }

__host__ __device__ constexpr int plane_buf(int nx, int ny, int nf, int np) {
  return (nf * odd_pad(np * plane_xlines(nx, ny)) > ny * odd_pad(np * (nx / 2 + 1)))
             ? nf * odd_pad(np * plane_xlines(nx, ny))
             : ny * odd_pad(np * (nx / 2 + 1));
}

__host__ __device__ constexpr size_t plane_lds_need(int nx, int ny, int nf, int np) {
  return sizeof(float2) * ((size_t)nx + ny + 2 * (size_t)plane_buf(nx, ny, nf, np));
}

size_t fft_plane_lds_bytes(int nx, int ny, int nf_x, int np) {
  const size_t b = plane_lds_need(nx, ny, nf_x, np);
  return b <= kPlaneLdsBudget ? b : 0;
}

// LDS budget of one plane workgroup: kPlaneLdsBudget for the full-size
// (kPlaneBlock-thread) workgroup, alone on its CU; half of it for the
// half-size one, two of which share a CU
__host__ __device__ constexpr size_t plane_budget(bool half) { return half ? kPlaneLdsBudget / 2 : kPlaneLdsBudget; }

// planes per workgroup of a batched plane launch allowing up to maxnp: the
// largest group whose buffers fit (the same on host and device)
__host__ __device__ inline int plane_group(int nx, int ny, int nf, int maxnp, bool half) {
  int g = maxnp;
  while (g > 1 && plane_lds_need(nx, ny, nf, g) > plane_budget(half)) g--;
  return g;
}

int plane_group_host(int nx, int ny, int nf, int maxnp, bool half) { return plane_group(nx, ny, nf, maxnp, half); }

bool plane_fits_half(int nx, int ny, int nf) { return plane_lds_need(nx, ny, nf, 1) <= plane_budget(true); }

// planes z .. z+np-1 of the real grid -> the same planes of the half spectrum
// (SPLIT: the y pass may use the split-precision matrix-core stage)
// Thread map of a row-major block of rows of w elements (w <= NT) for loops
// without a division per element: thread t takes column t mod w of rows
// t / w, t / w + step, ... with step = NT / w (threads past step * w idle).
struct ColMap {
  int c, r0, step;
  bool on;
};
template <int NT>
__device__ __forceinline__ ColMap col_map(int w) {
  ColMap m;
  m.step = NT / w;
  m.c = (int)threadIdx.x % w;
  m.r0 = (int)threadIdx.x / w;
  m.on = m.r0 < m.step;
  return m;
}

template <bool SPLIT, int NT>
__device__ __forceinline__ void fft_plane_fwd_body(const float* __restrict__ grid, float2* __restrict__ cg, int nx,
                                                   int ny, const AxisArgs& axx, const AxisArgs& axy, int z, int np,
                                                   float2* sm) {
  const int tid = threadIdx.x;
  const int nf = axx.rp.n;  // x line length: nx/2 (even nx) or nx
  const int hx = nx / 2 + 1;
  const int nrow = np * ny;                   // rows
  const int hyl = plane_xlines(nx, ny);      // x lines per plane
  const int nxl = np * hyl;                   // x lines
  const int ncol = np * hx;                   // y lines
  const int LSX = odd_pad(nxl), LSY = odd_pad(ncol);
  const int bsz = plane_buf(nx, ny, nf, np);
  float2* twx = sm;
  float2* twy = twx + nx;
  float2* b0 = twy + ny;
  float2* b1 = b0 + bsz;
  for (int i = tid; i < nx; i += NT) twx[i] = axx.tw[i];
  for (int i = tid; i < ny; i += NT) twy[i] = axy.tw[i];
  const bool even = (nx & 1) == 0;
  const size_t plane = (size_t)z * nx * ny;
  if (even) {
    const float2* src = reinterpret_cast<const float2*>(grid + plane);
    const ColMap m = col_map<NT>(nf);
    if (m.on)
      for (int rb = m.r0; rb < nrow; rb += kStageU * m.step) {
        float2 v[kStageU];
#pragma unroll
        for (int u = 0; u < kStageU; u++) {
          const int r = rb + u * m.step;
          v[u] = r < nrow ? src[(size_t)r * nf + m.c] : make_float2(0.f, 0.f);
        }
#pragma unroll
        for (int u = 0; u < kStageU; u++) {
          const int r = rb + u * m.step;
          if (r < nrow) b0[m.c * LSX + r] = v[u];
        }
      }
  } else {
    // rows 2j, 2j+1 of plane pl -> real and imaginary parts of x line
    // pl*hyl + j (an odd ny pairs the last row of each plane with zeros)
    const float* src = grid + plane;
    const SmallDiv dny = small_div(ny);
    const ColMap m = col_map<NT>(nx);
    if (m.on)
      for (int rb = m.r0; rb < nrow; rb += kStageU * m.step) {
        float v[kStageU];
#pragma unroll
        for (int u = 0; u < kStageU; u++) {
          const int r = rb + u * m.step;
          v[u] = r < nrow ? src[(size_t)r * nx + m.c] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < kStageU; u++) {
          const int r = rb + u * m.step;
          const int pl = sdiv(r, dny);
          const int y = r - pl * ny;
          if (r < nrow) reinterpret_cast<float*>(b0 + (m.c * LSX + pl * hyl + (y >> 1)))[y & 1] = v[u];
        }
      }
    if ((ny & 1) && m.on)
      for (int pl = m.r0; pl < np; pl += m.step) b0[m.c * LSX + pl * hyl + (ny >> 1)].y = 0.f;
  }
  __syncthreads();
  float2* res = fft_lines<-1>(b0, b1, twx, axx.rp, nxl, LSX, tid, NT);
  float2* q = res == b0 ? b1 : b0;
  // R2C post-processing (even nx) and transpose to columns:
  // X[k] = E[k] + w^k O[k], E = (Z[k] + Z*[h-k])/2, O = (Z[k] - Z*[h-k])/(2i)
  const SmallDiv dny = small_div(ny);
  const ColMap mh = col_map<NT>(hx);
  for (int r = mh.r0; mh.on && r < nrow; r += mh.step) {  // x line r (row of the plane group), point k
    const int k = mh.c;
    const int pl = sdiv(r, dny);
    const int y = r - pl * ny;
    float2 X;
    if (even) {
      const int h = nf;
      const float2 zk = res[(k == h ? 0 : k) * LSX + r];
      const float2 zc = cconj(res[(k == 0 ? 0 : h - k) * LSX + r]);
      const float2 E = cscale(cadd(zk, zc), 0.5f);
      const float2 D = csub(zk, zc);
      const float2 O = make_float2(0.5f * D.y, -0.5f * D.x);
      X = cadd(E, cmul(twx[k], O));
    } else {
      // Z = FFT(a + i b) of the row pair: A[k] = (Z[k] + Z*[nx-k]) / 2,
      // B[k] = (Z[k] - Z*[nx-k]) / (2i); row y is a (y even) or b (y odd)
      const int i = pl * hyl + (y >> 1);
      const float2 zk = res[k * LSX + i];
      const float2 zc = cconj(res[(k == 0 ? 0 : nx - k) * LSX + i]);
      const float2 D = csub(zk, zc);
      X = (y & 1) ? make_float2(0.5f * D.y, -0.5f * D.x) : cscale(cadd(zk, zc), 0.5f);
    }
    q[y * LSY + pl * hx + k] = X;
  }
  __syncthreads();
  float2* r2 = fft_lines<-1, SPLIT>(q, res, twy, axy.rp, ncol, LSY, tid, NT, axy.prec);
  const long long pz = spec_pitch(hx, ny);
  float2* dst = cg + (size_t)z * (size_t)pz;
  for (int r = mh.r0; mh.on && r < nrow; r += mh.step) {
    const int pl = sdiv(r, dny);
    const int y = r - pl * ny;
    dst[(size_t)pl * (size_t)pz + y * hx + mh.c] = r2[y * LSY + pl * hx + mh.c];
  }
}

// planes z .. z+np-1 of the half spectrum -> the same planes of the real grid
template <bool SPLIT, int NT>
__device__ __forceinline__ void fft_plane_inv_body(const float2* __restrict__ cg, float* __restrict__ grid, int nx,
                                                   int ny, const AxisArgs& axx, const AxisArgs& axy, int z, int np,
                                                   float2* sm) {
  const int tid = threadIdx.x;
  const int nf = axx.rp.n;
  const int hx = nx / 2 + 1;
  const int nrow = np * ny;                   // rows
  const int hyl = plane_xlines(nx, ny);      // x lines per plane
  const int nxl = np * hyl;                   // x lines
  const int ncol = np * hx;                   // y lines
  const int LSX = odd_pad(nxl), LSY = odd_pad(ncol);
  const int bsz = plane_buf(nx, ny, nf, np);
  float2* twx = sm;
  float2* twy = twx + nx;
  float2* b0 = twy + ny;
  float2* b1 = b0 + bsz;
  for (int i = tid; i < nx; i += NT) twx[i] = axx.tw[i];
  for (int i = tid; i < ny; i += NT) twy[i] = axy.tw[i];
  const long long pz = spec_pitch(hx, ny);
  const float2* src = cg + (size_t)z * (size_t)pz;
  const SmallDiv dny = small_div(ny);
  const ColMap mh = col_map<NT>(hx);
  if (mh.on)
    for (int rb = mh.r0; rb < nrow; rb += kStageU * mh.step) {
      float2 v[kStageU];
      int at[kStageU];  // LDS column offset of row r: y * LSY + pl * hx
#pragma unroll
      for (int u = 0; u < kStageU; u++) {
        const int r = rb + u * mh.step;
        const int pl = sdiv(r, dny);
        const int y = r - pl * ny;
        at[u] = y * LSY + pl * hx;
        v[u] = r < nrow ? src[(size_t)pl * (size_t)pz + y * hx + mh.c] : make_float2(0.f, 0.f);
      }
#pragma unroll
      for (int u = 0; u < kStageU; u++)
        if (rb + u * mh.step < nrow) b0[at[u] + mh.c] = v[u];
    }
  __syncthreads();
  float2* r = fft_lines<+1, SPLIT>(b0, b1, twy, axy.rp, ncol, LSY, tid, NT, axy.prec);
  float2* p = r == b0 ? b1 : b0;
  const bool even = (nx & 1) == 0;
  if (even) {
    // Z[k] = (X[k] + X*[h-k]) + i w^{-k} (X[k] - X*[h-k]),  k < h
    const int h = nf;
    const ColMap m = col_map<NT>(h);
    for (int row = m.r0; m.on && row < nrow; row += m.step) {
      const int k = m.c;
      const int pl = sdiv(row, dny);
      const float2* col = r + (row - pl * ny) * LSY + pl * hx;
      const float2 xk = col[k];
      const float2 xc = cconj(col[h - k]);
      const float2 A = cadd(xk, xc);
      const float2 B = cmul(cconj(twx[k]), csub(xk, xc));
      p[k * LSX + row] = make_float2(A.x - B.y, A.y + B.x);
    }
  } else {
    // x line pl*hyl + j: Z = A + i B from the full Hermitian spectra A, B of
    // rows 2j and 2j+1 of plane pl (zero past its last row); its inverse FFT
    // has row 2j in its real and row 2j+1 in its imaginary part
    const SmallDiv dhyl = small_div(hyl);
    const ColMap m = col_map<NT>(nx);
    for (int i = m.r0; m.on && i < nxl; i += m.step) {
      const int k = m.c;
      const int kk = k < hx ? k : nx - k;
      const int pl = sdiv(i, dhyl);
      const int ya = 2 * (i - pl * hyl);
      const float2* col = r + pl * hx + kk;
      float2 A = col[ya * LSY];
      float2 B = make_float2(0.f, 0.f);
      if (ya + 1 < ny) B = col[(ya + 1) * LSY];
      if (k >= hx) {
        A = cconj(A);
        B = cconj(B);
      }
      p[k * LSX + i] = make_float2(A.x - B.y, A.y + B.x);
    }
  }
  __syncthreads();
  float2* s = fft_lines<+1>(p, r, twx, axx.rp, nxl, LSX, tid, NT);
  const size_t plane = (size_t)z * nx * ny;
  if (even) {
    float2* dst = reinterpret_cast<float2*>(grid + plane);
    const ColMap m = col_map<NT>(nf);
    for (int row = m.r0; m.on && row < nrow; row += m.step) dst[(size_t)row * nf + m.c] = s[m.c * LSX + row];
  } else {
    float* dst = grid + plane;
    const ColMap m = col_map<NT>(nx);
    for (int row = m.r0; m.on && row < nrow; row += m.step) {
      const int pl = sdiv(row, dny);
      const int y = row - pl * ny;
      dst[(size_t)row * nx + m.c] = reinterpret_cast<const float*>(s + (m.c * LSX + pl * hyl + (y >> 1)))[y & 1];
    }
  }
}

template <bool SPLIT>
__global__ __launch_bounds__(kPlaneBlock) void k_fft_plane_fwd(const float* __restrict__ grid, float2* __restrict__ cg,
                                                              int nx, int ny, AxisArgs axx, AxisArgs axy) {
  extern __shared__ __align__(16) float2 sm[];
  fft_plane_fwd_body<SPLIT, kPlaneBlock>(grid, cg, nx, ny, axx, axy, blockIdx.x, 1, sm);
}

// Workgroup z < nz transforms plane z; with a pending energy/virial
// reduction the launch has one more workgroup that performs it alone (on a
// CU the planes leave free), so no plane's workgroup waits for it.
template <bool SPLIT>
__global__ __launch_bounds__(kPlaneBlock) void k_fft_plane_inv(const float2* __restrict__ cg, float* __restrict__ grid,
                                                              int nx, int ny, int nz, AxisArgs axx, AxisArgs axy,
                                                              EvReduce red) {
  extern __shared__ __align__(16) float2 sm[];
  if ((int)blockIdx.x >= nz) {
    ev_reduce_block<kPlaneBlock>(red);
    return;
  }
  fft_plane_inv_body<SPLIT, kPlaneBlock>(cg, grid, nx, ny, axx, axy, blockIdx.x, 1, sm);
}

hipError_t launch_fft_plane_fwd(const float* grid, float2* cg, int nx, int ny, int nz, const AxisArgs& ax,
                                const AxisArgs& ay, hipStream_t s) {
  const size_t lds = fft_plane_lds_bytes(nx, ny, ax.rp.n, 1);
  if (!lds) return hipErrorInvalidValue;
  if (ay.prec != PREC_FP32)
    hipLaunchKernelGGL(k_fft_plane_fwd<true>, dim3(nz), dim3(kPlaneBlock), lds, s, grid, cg, nx, ny, ax, ay);
  else
    hipLaunchKernelGGL(k_fft_plane_fwd<false>, dim3(nz), dim3(kPlaneBlock), lds, s, grid, cg, nx, ny, ax, ay);
  return hipGetLastError();
}

hipError_t launch_fft_plane_inv(const float2* cg, float* grid, int nx, int ny, int nz, const AxisArgs& ax,
                                const AxisArgs& ay, const EvReduce& red, hipStream_t s) {
  const size_t lds = fft_plane_lds_bytes(nx, ny, ax.rp.n, 1);
  if (!lds) return hipErrorInvalidValue;
  const dim3 g(nz + ((red.nsolve > 0 || red.nself > 0) ? 1 : 0));
  if (ay.prec != PREC_FP32)
    hipLaunchKernelGGL(k_fft_plane_inv<true>, g, dim3(kPlaneBlock), lds, s, cg, grid, nx, ny, nz, ax, ay, red);
  else
    hipLaunchKernelGGL(k_fft_plane_inv<false>, g, dim3(kPlaneBlock), lds, s, cg, grid, nx, ny, nz, ax, ay, red);
  return hipGetLastError();
}

// One tile of a y pass (S = -1 forward, +1 inverse) as a register four-step
// with n = N1 N2 in ONE LDS buffer: the first half loads its columns
// j2 + N2 j1 from HBM into registers, the second half reads its N2 points
// (k1 N2 + j2) back and stores X[k1 + N1 k2] straight to HBM (one LDS round
// trip instead of a staging copy and two).  Tile (tx, ty): lines
// kx0 = tx*TX ... of the hx lines at outer index ty.
template <int N1, int N2, int S>
__device__ __forceinline__ void cols_four_step(float2* __restrict__ cg, int hx, int TX, long long pt_stride,
                                               long long outer_stride, const AxisArgs& ax, int tx, int ty,
                                               float2* sm) {
  const int tid = threadIdx.x;
  float2* tw = sm;
  float2* b = sm + ax.ntw;
  for (int i = tid; i < ax.ntw; i += kBlock) tw[i] = ax.tw[i];
  const int ts = ax.rp.tstride;
  const int kx0 = tx * TX;
  const int nl = min(TX, hx - kx0);
  // the tile's first point (uniform) and 32-bit point offsets from it: a y
  // line spans n * pt_stride < 2^18 points (edges <= 512, pt_stride = hx)
  float2* __restrict__ tile = cg + ((size_t)kx0 + (size_t)ty * (size_t)outer_stride);
  const unsigned pst = (unsigned)pt_stride;
  const SmallDiv dtx = small_div(TX);
  for (int u0 = 0; u0 < N2 * TX; u0 += kBlock) {
    const int u = u0 + tid;
    const int j2 = sdiv(u, dtx);
    const int l = u - j2 * TX;
    const bool live = u < N2 * TX;
    float2 x[N1];
    const unsigned o = (unsigned)j2 * pst + (unsigned)l;
#pragma unroll
    for (int j1 = 0; j1 < N1; j1++)
      x[j1] = (live && l < nl) ? tile[o + (unsigned)(N2 * j1) * pst] : make_float2(0.f, 0.f);
    if (u0 == 0) __syncthreads();  // twiddles in LDS (uniform branch)
    if (live) {
      DftN<N1, S>::run(x);
      const int tj = mul24(j2, ts);
      b[j2 * TX + l] = x[0];
#pragma unroll
      for (int k1 = 1; k1 < N1; k1++) {
        float2 w = tw[k1 * tj];
        if (S > 0) w.y = -w.y;
        b[(k1 * N2 + j2) * TX + l] = cmul(x[k1], w);
      }
    }
  }
  __syncthreads();
  for (int u = tid; u < N1 * TX; u += kBlock) {
    const int k1 = sdiv(u, dtx);
    const int l = u - k1 * TX;
    float2 X[N2];
#pragma unroll
    for (int j2 = 0; j2 < N2; j2++) X[j2] = b[(k1 * N2 + j2) * TX + l];
    DftN<N2, S>::run(X);
    if (l < nl) {
      const unsigned o = (unsigned)k1 * pst + (unsigned)l;
#pragma unroll
      for (int k2 = 0; k2 < N2; k2++) tile[o + (unsigned)(N1 * k2) * pst] = X[k2];
    }
  }
}

// the y pass of a tile through cols_four_step for the pair of code
template <int S>
__device__ __forceinline__ void cols_four_step_dispatch(int code, float2* __restrict__ cg, int hx, int TX,
                                                        long long pt_stride, long long outer_stride,
                                                        const AxisArgs& ax, int tx, int ty, float2* sm) {
  switch (code) {
#define PME_YC_CASE(c, a, b) \
  case c: cols_four_step<a, b, S>(cg, hx, TX, pt_stride, outer_stride, ax, tx, ty, sm); break;
    PME_F4_PAIRS(PME_YC_CASE)
#undef PME_YC_CASE
    default: break;
  }
}

// ------------------------------------------------------------ y / z passes --

// Column tile (tx, ty) of one grid: lines kx0 = tx*TX ... of the hx lines at
// outer index ty.  The y pass: hx = nx/2 + 1 columns per (kz = ty).  The z
// pass: hx = the hxd * ny lines of a z plane, flattened (ky, kx) with rows of
// hxd = nx/2 + 1, and ty = 0.  blk indexes the energy/virial partial of the
// tile.
template <int MODE, bool SPLIT>
__device__ __forceinline__ void fft_cols_body(float2* __restrict__ cg, int n, int hx, int TX, long long pt_stride,
                                              long long outer_stride, const AxisArgs& ax, const SolveArgs& sa,
                                              int tx, int ty, int blk, float2* sm, int hxd) {
  // y passes with a four-step pair (ax.f4col, set for the y axis when the pair
  // is the radix plan's): one LDS buffer, columns straight from and to HBM
  if ((MODE == COL_FWD || MODE == COL_INV) && !SPLIT && ax.f4col >= 0) {
    cols_four_step_dispatch<MODE == COL_FWD ? -1 : 1>(ax.f4col, cg, hx, TX, pt_stride, outer_stride, ax, tx, ty, sm);
    return;
  }
  __shared__ double sh_red[7 * (kBlock / 64)];
  const int tid = threadIdx.x;
  float2* tw = sm;
  float2* b0 = sm + ax.ntw;
  float2* b1 = b0 + n * TX;
  for (int i = tid; i < ax.ntw; i += kBlock) tw[i] = ax.tw[i];
  const int kx0 = tx * TX;
  const int nl = min(TX, hx - kx0);
  const size_t base = (size_t)kx0 + (size_t)ty * (size_t)outer_stride;
  for (int e0 = tid; e0 < n * TX; e0 += kStageU * kBlock) {
    float2 v[kStageU];
#pragma unroll
    for (int u = 0; u < kStageU; u++) {
      const int e = e0 + u * kBlock;
      const int j = sdiv(e, small_div(TX));
      const int l = e - j * TX;
      v[u] = (e < n * TX && l < nl) ? cg[base + (size_t)j * pt_stride + l] : make_float2(0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < kStageU; u++) {
      const int e = e0 + u * kBlock;
      if (e < n * TX) b0[e] = v[u];
    }
  }
  __syncthreads();
  float2* res;
  if (MODE == COL_INV) {
    res = fft_lines<+1, SPLIT>(b0, b1, tw, ax.rp, TX, TX, tid, kBlock, ax.prec);
  } else {
    res = fft_lines<-1, SPLIT>(b0, b1, tw, ax.rp, TX, TX, tid, kBlock, ax.prec);
  }
  double acc[7] = {0, 0, 0, 0, 0, 0, 0};
  if (MODE == COL_FWD_SOLVE_INV) {
    solve_lines(sa, res, n, TX, nl, kx0, hxd, acc);
    __syncthreads();
  }
  if (MODE == COL_FWD_SOLVE_INV || MODE == COL_FWD_INV) {
    res = fft_lines<+1, SPLIT>(res, res == b0 ? b1 : b0, tw, ax.rp, TX, TX, tid, kBlock, ax.prec);
  }
  for (int e = tid; e < n * TX; e += kBlock) {
    const int j = sdiv(e, small_div(TX));
    const int l = e - j * TX;
    if (l < nl) cg[base + (size_t)j * pt_stride + l] = res[e];
  }
  if (MODE == COL_FWD_SOLVE_INV && sa.calc_ev) ev_partial(sa, acc, sh_red, blk);
}

template <int MODE, bool SPLIT>
__global__ __launch_bounds__(kBlock) void k_fft_cols(float2* __restrict__ cg, int n, int hx, int TX,
                                                     long long pt_stride, long long outer_stride, AxisArgs ax,
                                                     SolveArgs sa, EvReduce red, int hxd) {
  extern __shared__ __align__(16) float2 sm[];
  if ((red.nsolve > 0 || red.nself > 0) && blockIdx.x == 0 && blockIdx.y == 0) ev_reduce_block<kBlock>(red);
  fft_cols_body<MODE, SPLIT>(cg, n, hx, TX, pt_stride, outer_stride, ax, sa, blockIdx.x, blockIdx.y,
                      blockIdx.x + gridDim.x * blockIdx.y, sm, hxd);
}

// Stand-alone scalar sum over the whole half spectrum (used when the spectrum
// has been materialised, e.g. scalar_sum called twice, and for a triclinic box
// whose z length has no four-step pair or runs in split precision).
__global__ __launch_bounds__(kBlock) void k_scalar_sum(float2* __restrict__ cg, int hx, int total, SolveArgs sa) {
  __shared__ double sh_red[7 * (kBlock / 64)];
  double acc[7] = {0, 0, 0, 0, 0, 0, 0};
  const int idx = blockIdx.x * kBlock + threadIdx.x;
  if (idx < total) {
    const int k1 = idx % hx;
    const int t = idx / hx;
    const int k2 = t % sa.n2;
    const int k3 = t / sa.n2;
    const size_t a = (size_t)k3 * (size_t)spec_pitch(hx, sa.n2) + (size_t)k2 * hx + k1;
    cg[a] = sa.tric ? solve_point_tric(sa, cg[a], k1, k2, k3, acc) : solve_point(sa, cg[a], k1, k2, k3, acc);
  }
  if (sa.calc_ev) ev_partial(sa, acc, sh_red, blockIdx.x);
}

// ----------------------------------------------------------------- launch --

size_t fft_x_lds_bytes(int nf, int NR, int ntw) { return sizeof(float2) * ((size_t)ntw + 2 * (size_t)nf * (NR + 1)); }
size_t fft_cols_lds_bytes(int n, int TX, int nbuf) { return sizeof(float2) * ((size_t)n + (size_t)nbuf * n * TX); }

hipError_t launch_fft_x_r2c(const float* grid, float2* cg, int nx, int ny, int nz, int NR, const AxisArgs& ax,
                            hipStream_t s) {
  const size_t lds = fft_x_lds_bytes(ax.rp.n, NR, ax.ntw);
  const int nrows = ny * nz;
  hipLaunchKernelGGL(k_fft_x_r2c, dim3((nrows + NR - 1) / NR), dim3(kBlock), lds, s, grid, cg, nx, nrows, ny, NR,
                     ax);
  return hipGetLastError();
}

hipError_t launch_fft_x_c2r(const float2* cg, float* grid, int nx, int ny, int nz, int NR, const AxisArgs& ax,
                            hipStream_t s) {
  const size_t lds = fft_x_lds_bytes(ax.rp.n, NR, ax.ntw);
  const int nrows = ny * nz;
  hipLaunchKernelGGL(k_fft_x_c2r, dim3((nrows + NR - 1) / NR), dim3(kBlock), lds, s, cg, grid, nx, nrows, ny, NR,
                     ax);
  return hipGetLastError();
}

int cols_blocks(int hx, int TX, int nouter) { return ((hx + TX - 1) / TX) * nouter; }

hipError_t launch_fft_cols(int mode, float2* cg, int n, int hx, int TX, long long pt_stride, int nouter,
                           long long outer_stride, const AxisArgs& ax, const SolveArgs& sa, const EvReduce& red,
                           int hxd, hipStream_t s) {
  const bool split = ax.prec != PREC_FP32;
  const bool four_step = mode == COL_FWD_SOLVE_INV && !split && ax.f4 >= 0;
  const bool split_four_step = mode == COL_FWD_SOLVE_INV && split && ax.rp.f4a == 16;
  const size_t lds = fft_cols_lds_bytes(n, TX, four_step || split_four_step ? 1 : 2);
  const dim3 grid((hx + TX - 1) / TX, nouter);
  // the fused z pass indexes its tile with shifts
  if (mode == COL_FWD_SOLVE_INV && sa.tric && !four_step) return hipErrorInvalidValue;  // no such kernel
  if (mode == COL_FWD_SOLVE_INV && (TX <= 0 || (TX & (TX - 1)) != 0)) return hipErrorInvalidValue;
  if (four_step) {
    if (nouter != 1 || outer_stride != 0) return hipErrorInvalidValue;  // one flattened plane of lines
    return launch_zsolve(cg, hx, TX, pt_stride, ax, sa, red, hxd, lds, s);
  }
  if (split_four_step) {
    if (nouter != 1 || outer_stride != 0) return hipErrorInvalidValue;
    return launch_zsolve_split(cg, hx, TX, pt_stride, ax, sa, red, hxd, lds, s);
  }
#define PME_COLS(M)                                                                                         \
  if (split)                                                                                              \
    hipLaunchKernelGGL((k_fft_cols<M, true>), grid, dim3(kBlock), lds, s, cg, n, hx, TX, pt_stride, outer_stride, ax, sa, red, hxd); \
  else                                                                                                    \
    hipLaunchKernelGGL((k_fft_cols<M, false>), grid, dim3(kBlock), lds, s, cg, n, hx, TX, pt_stride, outer_stride, ax, sa, red, hxd);
  switch (mode) {
    case COL_FWD: PME_COLS(COL_FWD); break;
    case COL_INV: PME_COLS(COL_INV); break;
    case COL_FWD_SOLVE_INV: PME_COLS(COL_FWD_SOLVE_INV); break;
    case COL_FWD_INV: PME_COLS(COL_FWD_INV); break;
    default:
      return hipErrorInvalidValue;
  }
#undef PME_COLS
  return hipGetLastError();
}

int scalar_sum_blocks(int total) { return (total + kBlock - 1) / kBlock; }

hipError_t launch_scalar_sum(float2* cg, int hx, const SolveArgs& sa, hipStream_t s) {
  const int total = hx * sa.n2 * sa.n3;
  hipLaunchKernelGGL(k_scalar_sum, dim3((total + kBlock - 1) / kBlock), dim3(kBlock), 0, s, cg, hx, total, sa);
  return hipGetLastError();
}

// ---- batched: persistent workgroups over the work items of many systems ----

template <int INV>
__global__ __launch_bounds__(kBlock) void k_batch_fft_x(const SysDesc* __restrict__ sys,
                                                        const WorkItem* __restrict__ items, int nitems) {
  extern __shared__ __align__(16) float2 sm[];
  for (int it = blockIdx.x; it < nitems; it += gridDim.x) {
    const WorkItem w = uniform_item(items[it]);
    const SysDesc& d = sys[w.sys];
    const int nrows = d.bin.ny * d.bin.nz;
    if (INV)
      fft_x_c2r_body(d.cgrid, d.grid, d.bin.nx, nrows, d.bin.ny, d.NR, d.ax[0], w.idx, sm);
    else
      fft_x_r2c_body(d.grid, d.cgrid, d.bin.nx, nrows, d.bin.ny, d.NR, d.ax[0], w.idx, sm);
    __syncthreads();
  }
}

// the fused z pass of a split-precision axis of 16 f4b points (a single
// system's: k_zsolve_split)
__device__ __forceinline__ void zsolve_split_dispatch(float2* __restrict__ cg, int hx, int TX, long long pt_stride,
                                                      const AxisArgs& ax, const SolveArgs& sa, int blk, float2* sm,
                                                      int hxd) {
  switch (ax.rp.f4b) {
#define PME_ZS_SPLIT(L)                                                                                  \
  case L:                                                                                                \
    if (ax.prec == PREC_BF16X3)                                                                          \
      zsolve_four_step_split<L, PREC_BF16X3>(cg, hx, TX, pt_stride, 0, ax, sa, blk, 0, blk, sm, hxd);    \
    else                                                                                                 \
      zsolve_four_step_split<L, PREC_FP16X3>(cg, hx, TX, pt_stride, 0, ax, sa, blk, 0, blk, sm, hxd);    \
    break;
    PME_ZSOLVE_SPLIT_LENGTHS(PME_ZS_SPLIT)
#undef PME_ZS_SPLIT
    default: break;
  }
}

// split z passes: held to three waves per SIMD (the compiler takes 256 VGPRs
// for the union of the lengths, one wave; 22 are spilled).  24 systems of 48 to 96 points, planes
// included: 286 -> 207 us per solve (211 with the 16-point DFT first in the inverse).
template <int AXIS, int MODE, bool SPLIT>
__global__ __launch_bounds__(kBlock, AXIS == 2 && SPLIT ? 3 : 1) void k_batch_cols(const SysDesc* __restrict__ sys,
                                                       const WorkItem* __restrict__ items, int nitems, int reduce) {
  extern __shared__ __align__(16) float2 sm[];
  for (int it = blockIdx.x; it < nitems; it += gridDim.x) {
    const WorkItem w = uniform_item(items[it]);
    const SysDesc& d = sys[w.sys];
    if (reduce && w.idx == 0 && (d.sa.calc_ev || d.calc_self)) batch_ev_reduce<kBlock>(d);
    const int hx = d.bin.nx / 2 + 1;
    const long long pz = spec_pitch(hx, d.bin.ny);
    if (AXIS == 1) {  // y: tiles of kx per kz
      const int ntx = (hx + d.TXy - 1) / d.TXy;
      fft_cols_body<MODE, SPLIT>(d.cgrid, d.bin.ny, hx, d.TXy, hx, pz, d.ax[1], d.sa, w.idx % ntx, w.idx / ntx,
                                 w.idx, sm, hx);
    } else if (SPLIT && MODE == COL_FWD_SOLVE_INV && d.ax[2].rp.f4a == 16 && d.ax[2].prec != PREC_FP32) {
      zsolve_split_dispatch(d.cgrid, hx * d.bin.ny, d.TXz, pz, d.ax[2], d.sa, w.idx, sm, hx);
    } else {  // z: tiles of the flattened (ky, kx) of a plane
      fft_cols_body<MODE, SPLIT>(d.cgrid, d.bin.nz, hx * d.bin.ny, d.TXz, pz, 0, d.ax[2], d.sa, w.idx, 0, w.idx, sm,
                                 hx);
    }
    __syncthreads();
  }
}

// items are (system, first plane z); each covers planes z .. z+g-1 with g =
// plane_group(.., maxnp, NT < kPlaneBlock) of its system (fewer at the top of
// the grid).  SPLIT: every system of the launch may use the matrix-core stage
// in y.  NT = kPlaneBlock / 2: half-size workgroups, two per CU, for the
// systems whose plane fits half the LDS budget: one workgroup's HBM loads and
// stores then overlap the other's transforms.
template <int INV, bool SPLIT, int NT>
__global__ __launch_bounds__(NT, 4) void k_batch_plane(const SysDesc* __restrict__ sys,
                                                    const WorkItem* __restrict__ items, int nitems, int reduce,
                                                    int maxnp) {
  extern __shared__ __align__(16) float2 sm[];
  for (int it = blockIdx.x; it < nitems; it += gridDim.x) {
    const WorkItem w = uniform_item(items[it]);
    const SysDesc& d = sys[w.sys];
    const int npl = min(plane_group(d.bin.nx, d.bin.ny, d.ax[0].rp.n, maxnp, NT < kPlaneBlock), d.bin.nz - w.idx);
    if (INV) {
      if (reduce && w.idx == 0 && (d.sa.calc_ev || d.calc_self)) batch_ev_reduce<NT>(d);
      fft_plane_inv_body<SPLIT, NT>(d.cgrid, d.grid, d.bin.nx, d.bin.ny, d.ax[0], d.ax[1], w.idx, npl, sm);
    } else {
      fft_plane_fwd_body<SPLIT, NT>(d.grid, d.cgrid, d.bin.nx, d.bin.ny, d.ax[0], d.ax[1], w.idx, npl, sm);
    }
    __syncthreads();
  }
}

hipError_t launch_batch_plane(int inverse, int reduce, int maxnp, int split, int half, const SysDesc* sys,
                              const WorkItem* items, int nitems, int grid, size_t lds, hipStream_t s) {
  if (nitems <= 0) return hipSuccess;
  if (maxnp < 1 || maxnp > kPlaneGroupMax) return hipErrorInvalidValue;
  const dim3 g(grid);
#define PME_BPLANE(I, S)                                                                                        \
  if (half)                                                                                                     \
    hipLaunchKernelGGL((k_batch_plane<I, S, kPlaneBlock / 2>), g, dim3(kPlaneBlock / 2), lds, s, sys, items,   \
                       nitems, reduce, maxnp);                                                                  \
  else                                                                                                          \
    hipLaunchKernelGGL((k_batch_plane<I, S, kPlaneBlock>), g, dim3(kPlaneBlock), lds, s, sys, items, nitems,    \
                       reduce, maxnp);
  if (inverse && split) {
    PME_BPLANE(1, true)
  } else if (inverse) {
    PME_BPLANE(1, false)
  } else if (split) {
    PME_BPLANE(0, true)
  } else {
    PME_BPLANE(0, false)
  }
#undef PME_BPLANE
  return hipGetLastError();
}

hipError_t launch_batch_fft_x(int inverse, const SysDesc* sys, const WorkItem* items, int nitems, int grid, size_t lds,
                              hipStream_t s) {
  if (nitems <= 0) return hipSuccess;
  if (inverse)
    hipLaunchKernelGGL(k_batch_fft_x<1>, dim3(grid), dim3(kBlock), lds, s, sys, items, nitems);
  else
    hipLaunchKernelGGL(k_batch_fft_x<0>, dim3(grid), dim3(kBlock), lds, s, sys, items, nitems);
  return hipGetLastError();
}

hipError_t launch_batch_cols(int axis, int mode, int reduce, int split, const SysDesc* sys, const WorkItem* items,
                             int nitems, int grid, size_t lds, hipStream_t s) {
  if (nitems <= 0) return hipSuccess;
  const dim3 g(grid), b(kBlock);
#define PME_BCOLS(A, M)                                                                                 \
  if (split)                                                                                          \
    hipLaunchKernelGGL((k_batch_cols<A, M, true>), g, b, lds, s, sys, items, nitems, reduce);         \
  else                                                                                                \
    hipLaunchKernelGGL((k_batch_cols<A, M, false>), g, b, lds, s, sys, items, nitems, reduce);
  if (axis == 1 && mode == COL_FWD) { PME_BCOLS(1, COL_FWD); }
  else if (axis == 1 && mode == COL_INV) { PME_BCOLS(1, COL_INV); }
  else if (axis == 2 && mode == COL_FWD_SOLVE_INV) { PME_BCOLS(2, COL_FWD_SOLVE_INV); }
  else return hipErrorInvalidValue;
#undef PME_BCOLS
  return hipGetLastError();
}

}  // namespace pme
