// pme_plane.hip -- x and y transforms of whole z planes as register four-step
// FFTs in one LDS buffer.
//
// A workgroup transforms np consecutive z planes of the grid.  Both line
// lengths (x: nx/2 complex points for even nx, nx for odd; y: ny) factor as
// A B with codelet lengths, so a line transform is two passes over registers
// (DFT_A, twiddle, DFT_B) and the whole plane is four:
//
//   forward   1  HBM rows -> DFT_Ax -> LDS         (real rows as x lines)
//             2  LDS -> DFT_Bx -> LDS, in place
//             3  LDS -> R2C split of a (k, h-k) pair of columns, DFT_Ay -> LDS, in place
//             4  LDS -> DFT_By -> HBM half-spectrum plane
//   inverse   1  HBM half-spectrum plane -> DFT_Ay -> LDS
//             2  LDS -> DFT_By, C2R merge of a (k, h-k) pair -> LDS, in place
//             3  LDS -> DFT_Ax -> LDS, in place
//             4  LDS -> DFT_Bx -> HBM real rows
//
// Each plane is read and written once and makes three LDS round trips
// with three barriers; staging copies, the transposition and the R2C/C2R
// passes have no round trip of their own.  Every middle pass rewrites exactly
// the points it read, so ONE buffer of (nx/2 + 1) ny points serves (odd nx: the
// pair split mixes rows, so the spectrum columns have a buffer of their own).
// A plane of 144 x 144 takes 84 KB of the 160 KB LDS.
//
// A split-precision y axis of 16 b points (b a codelet length up to 12) takes
// DFT_Ay = 16 and DFT_By = b in both directions and runs the 16-point DFTs on the
// matrix cores (SPLIT).  They come first forward too: after the other factor their
// columns mix large and small frequencies, and the hi-lo error, which goes with the
// column's largest, was 15 % more in the forces.
//
// Bound by the VALU and the LDS round trips, not by HBM (the two launches of
// the 108 x 100 x 96 grid move 16 MB).  LDS points are line-minor (point p of
// line l at p * LS + l, LS odd): lanes run along lines in the passes that
// read or write LDS only, along consecutive points in those that touch HBM.
#include <algorithm>

#include "pme_internal.hpp"

namespace pme {

// codelet lengths of the plane passes
#define PME_PL_LENGTHS(X) X(2) X(3) X(4) X(5) X(6) X(8) X(9) X(10) X(12) X(15) X(16)
// those of the passes that hold two columns in registers (the smaller y factor)
#define PME_PL_PAIR_MAX 12
#define PME_PL_PAIR_LENGTHS(X) X(2) X(3) X(4) X(5) X(6) X(8) X(9) X(10) X(12)
#define PME_PL_PAIR_SWITCH(len, CALL)  \
  switch (len) {                       \
    PME_PL_PAIR_LENGTHS(CALL)          \
    default: break;                    \
  }
#define PME_PL_SWITCH(len, CALL)       \
  switch (len) {                       \
    PME_PL_LENGTHS(CALL)               \
    default: break;                    \
  }

// Geometry of a plane group (the same on host and device)
struct PlaneGeo {
  int nx, ny, np;
  int h;        // x line length
  int hx;       // spectrum columns of a plane
  int nxl;      // x lines of the group
  int LX, LY;   // LDS line pitch of the x lines and of the columns' rows
  bool odd;
  int bx, by;   // points of the x-line buffer, of the separate column buffer (odd nx)
};
__host__ __device__ __forceinline__ PlaneGeo plane_geo(int nx, int ny, int np) {
  PlaneGeo g;
  g.nx = nx;
  g.ny = ny;
  g.np = np;
  g.odd = (nx & 1) != 0;
  g.h = g.odd ? nx : nx >> 1;
  g.hx = nx / 2 + 1;
  g.nxl = np * (g.odd ? (ny + 1) >> 1 : ny);
  g.LX = g.nxl | 1;
  g.LY = (np * ny) | 1;
  g.bx = g.odd ? nx * g.LX : g.hx * g.LY;  // even: LX == LY and one spare column for k = nx/2
  g.by = g.odd ? g.hx * g.LY : 0;
  return g;
}

size_t plane4_lds_need(int nx, int ny, int np) {
  const PlaneGeo g = plane_geo(nx, ny, np);
  return sizeof(float2) * ((size_t)nx + ny + g.bx + g.by);
}

bool plane4_ok(const RadixPlan& rx, const RadixPlan& ry) { return rx.f4a > 0 && ry.f4a > 0 && ry.f4a <= PME_PL_PAIR_MAX; }

// split-precision y axis: 16 b with the 16-point DFTs on the matrix cores, b
// the smaller factor's codelet
static bool plane4_split_ok(const RadixPlan& rx, const RadixPlan& ry) {
  return rx.f4a > 0 && ry.f4a == 16 && ry.f4b > 0 && ry.f4b <= PME_PL_PAIR_MAX;
}

size_t fft_plane4_lds_bytes(int nx, int ny, int np) {
  const size_t b = plane4_lds_need(nx, ny, np);
  return b <= kPlaneLdsBudget ? b : 0;
}

PlaneKind plane_kind(int nx, int ny, const RadixPlan& rx, const RadixPlan& ry, int y_prec) {
  if (fft_plane4_lds_bytes(nx, ny, 1)) {
    if (y_prec == PREC_FP32 && plane4_ok(rx, ry)) return PLANE_FOUR_STEP;
    if (y_prec != PREC_FP32 && plane4_split_ok(rx, ry)) return PLANE_FOUR_STEP_SPLIT;
  }
  return fft_plane_lds_bytes(nx, ny, rx.n, 1) ? PLANE_STAGES : PLANE_NONE;
}

__device__ __forceinline__ int plane4_group(int nx, int ny, int maxnp, bool half) {
  const size_t budget = half ? kPlaneLdsBudget / 2 : kPlaneLdsBudget;
  int np = maxnp;
  while (np > 1) {
    const PlaneGeo g = plane_geo(nx, ny, np);
    if (sizeof(float2) * ((size_t)nx + ny + g.bx + g.by) <= budget) break;
    np--;
  }
  return np;
}
int plane4_group_host(int nx, int ny, int maxnp, bool half) {
  const size_t budget = half ? kPlaneLdsBudget / 2 : kPlaneLdsBudget;
  int np = maxnp;
  while (np > 1 && plane4_lds_need(nx, ny, np) > budget) np--;
  return np;
}
bool plane4_fits_half(int nx, int ny) { return plane4_lds_need(nx, ny, 1) <= kPlaneLdsBudget / 2; }

__device__ __forceinline__ float2 cmulc(float2 a, float2 b) { return cmul(a, cconj(b)); }

// ---- passes shared by both directions ------------------------------------------

// DFT_B over j2 of the points (k1 B + j2) of every line, in place: unit (k1, l)
template <int B, int S, int NT>
__device__ __forceinline__ void pl_dft_b(float2* b, int A, int nl, int LS) {
  const SmallDiv dl = small_div(nl);
  for (int u = threadIdx.x; u < A * nl; u += NT) {
    const int k1 = sdiv(u, dl);
    float2* p = b + mul24(mul24(k1, B), LS) + (u - mul24(k1, nl));
    float2 x[B];
#pragma unroll
    for (int j = 0; j < B; j++) x[j] = p[mul24(j, LS)];
    DftN<B, S>::run(x);
#pragma unroll
    for (int j = 0; j < B; j++) p[mul24(j, LS)] = x[j];
  }
}

// DFT_A over j1 of the points (j2 + B j1) of every line, times w^{S j2 k1},
// in place: unit (j2, l)
template <int A, int S, int NT>
__device__ __forceinline__ void pl_dft_a(float2* b, const float2* tw, int tstride, int B, int nl, int LS) {
  const SmallDiv dl = small_div(nl);
  const int BLS = mul24(B, LS);
  for (int u = threadIdx.x; u < B * nl; u += NT) {
    const int j2 = sdiv(u, dl);
    float2* p = b + mul24(j2, LS) + (u - mul24(j2, nl));
    const int ts = mul24(j2, tstride);
    float2 x[A];
#pragma unroll
    for (int j = 0; j < A; j++) x[j] = p[mul24(j, BLS)];
    DftN<A, S>::run(x);
    p[0] = x[0];
#pragma unroll
    for (int k = 1; k < A; k++) {
      const float2 w = tw[mul24(k, ts)];
      p[mul24(k, BLS)] = S < 0 ? cmul(x[k], w) : cmulc(x[k], w);
    }
  }
}

// ---- forward ---------------------------------------------------------------------

// pass 1: unit (x line, j2), j2 fastest (runs of B points of a row), points
// j2 + B j1 from HBM.  Odd nx: rows 2j, 2j+1 of a plane are the real and
// imaginary parts of one line (an odd ny pairs the last row with zeros).
template <int A, int NT>
__device__ __forceinline__ void pl_fwd_load(const float* __restrict__ src, float2* b, const float2* tw, int tstride,
                                            int B, const PlaneGeo& g) {
  const SmallDiv dB = small_div(B);
  const int hyl = (g.ny + 1) >> 1;
  const SmallDiv dh = small_div(hyl);
  const int n = g.nxl * B;
  const int BLS = mul24(B, g.LX);
  for (int u0 = 0; u0 < n; u0 += NT) {
    const int u = u0 + (int)threadIdx.x;
    const int l = sdiv(u, dB);
    const int j2 = u - mul24(l, B);
    const bool live = u < n;
    float2 x[A];
    if (!g.odd) {
      const float2* s = reinterpret_cast<const float2*>(src) + (mul24(l, g.h) + j2);
#pragma unroll
      for (int j = 0; j < A; j++) x[j] = live ? s[mul24(j, B)] : make_float2(0.f, 0.f);
    } else {
      const int pl = sdiv(l, dh);
      const int y = 2 * (l - mul24(pl, hyl));
      const float* s = src + (mul24(mul24(pl, g.ny) + y, g.nx) + j2);
      const bool two = y + 1 < g.ny;
#pragma unroll
      for (int j = 0; j < A; j++) {
        x[j].x = live ? s[mul24(j, B)] : 0.f;
        x[j].y = live && two ? s[mul24(j, B) + g.nx] : 0.f;
      }
    }
    if (u0 == 0) __syncthreads();  // twiddles in LDS (uniform branch)
    if (live) {
      DftN<A, -1>::run(x);
      float2* p = b + (mul24(j2, g.LX) + l);
      const int ts = mul24(j2, tstride);
      p[0] = x[0];
#pragma unroll
      for (int k = 1; k < A; k++) p[mul24(k, BLS)] = cmul(x[k], tw[mul24(k, ts)]);
    }
  }
}

// pass 3, even nx: unit (pair k <= h/2, plane, j2), j2 fastest: Z[k] and
// Z[h-k] of the rows j2 + B j1 give columns k and h-k of the half spectrum
//   X[k] = E + w^k O, X[h-k] = conj(E - w^k O),
//   E = (Z[k] + Z*[h-k])/2, O = (Z[k] - Z*[h-k])/(2i)
// (k = 0 pairs with column h, stored in the spare slot), then DFT_A and the
// twiddle over the rows.  x point k sits at slot (k mod Ax) Bx + k / Ax.
template <int A, int NT>
__device__ __forceinline__ void pl_fwd_split(float2* b, const float2* twx, const float2* twy, int B, int Ax, int Bx,
                                             const PlaneGeo& g) {
  const SmallDiv dB = small_div(B), dnp = small_div(g.np), dax = small_div(Ax);
  const int n = mul24(mul24((g.h >> 1) + 1, g.np), B);
  for (int u = threadIdx.x; u < n; u += NT) {
    const int t = sdiv(u, dB);
    const int j2 = u - mul24(t, B);
    const int k = sdiv(t, dnp);
    const int r = mul24(t - mul24(k, g.np), g.ny) + j2;
    const int c = g.h - k;
    const int qk = sdiv(k, dax), qc = sdiv(c, dax);
    float2* pk = b + (mul24(mul24(k - mul24(qk, Ax), Bx) + qk, g.LX) + r);
    float2* pc = b + (mul24(k == 0 ? g.h : mul24(c - mul24(qc, Ax), Bx) + qc, g.LX) + r);
    const float2* pz = k == 0 ? pk : pc;
    const float2 w = twx[k];
    float2 xk[A], xc[A];
#pragma unroll
    for (int j = 0; j < A; j++) {
      xk[j] = pk[mul24(j, B)];
      xc[j] = pz[mul24(j, B)];
    }
#pragma unroll
    for (int j = 0; j < A; j++) {
      const float2 zc = cconj(xc[j]);
      const float2 E = cscale(cadd(xk[j], zc), 0.5f);
      const float2 D = csub(xk[j], zc);
      const float2 T = cmul(w, make_float2(0.5f * D.y, -0.5f * D.x));
      xk[j] = cadd(E, T);
      xc[j] = cconj(csub(E, T));
    }
    DftN<A, -1>::run(xk);
    DftN<A, -1>::run(xc);
    pk[0] = xk[0];
    if (c != k) pc[0] = xc[0];
#pragma unroll
    for (int q = 1; q < A; q++) {
      const float2 wy = twy[mul24(q, j2)];
      pk[mul24(q, B)] = cmul(xk[q], wy);
      if (c != k) pc[mul24(q, B)] = cmul(xc[q], wy);
    }
  }
}

// pass 3, odd nx: unit (column k, plane, j2): row y is the real (y even) or
// imaginary (y odd) row of line y/2: A[k] = (Z[k] + Z*[nx-k])/2, B[k] = (Z[k] -
// Z*[nx-k])/(2i); into the column buffer
template <int A, int NT>
__device__ __forceinline__ void pl_fwd_pair(const float2* b, float2* d, const float2* twy, int B, int Ax, int Bx,
                                            const PlaneGeo& g) {
  const SmallDiv dB = small_div(B), dnp = small_div(g.np), dax = small_div(Ax);
  const int hyl = (g.ny + 1) >> 1;
  const int n = mul24(mul24(g.hx, g.np), B);
  for (int u = threadIdx.x; u < n; u += NT) {
    const int t = sdiv(u, dB);
    const int j2 = u - mul24(t, B);
    const int k = sdiv(t, dnp);
    const int pl = t - mul24(k, g.np);
    const int c = k == 0 ? 0 : g.nx - k;
    const int qk = sdiv(k, dax), qc = sdiv(c, dax);
    const float2* pk = b + (mul24(mul24(k - mul24(qk, Ax), Bx) + qk, g.LX) + mul24(pl, hyl));
    const float2* pc = b + (mul24(mul24(c - mul24(qc, Ax), Bx) + qc, g.LX) + mul24(pl, hyl));
    float2 x[A];
#pragma unroll
    for (int j = 0; j < A; j++) {
      const int y = j2 + mul24(j, B);
      const float2 zk = pk[y >> 1], zc = cconj(pc[y >> 1]);
      const float2 D = csub(zk, zc);
      x[j] = (y & 1) ? make_float2(0.5f * D.y, -0.5f * D.x) : cscale(cadd(zk, zc), 0.5f);
    }
    DftN<A, -1>::run(x);
    float2* p = d + (mul24(k, g.LY) + mul24(pl, g.ny) + j2);
    p[0] = x[0];
#pragma unroll
    for (int q = 1; q < A; q++) p[mul24(q, B)] = cmul(x[q], twy[mul24(q, j2)]);
  }
}

// pass 3 with the DFT_16 as hi-lo products on the matrix cores, even nx: 32
// columns per wave are 16 units (pair, plane, j2), lanes j and j + 16 columns k and
// h-k of one unit, each forming its own column of the split as it loads.  In place:
// a wave has loaded all its columns before it stores the first.
template <int PREC, int NT>
__device__ __forceinline__ void pl_fwd_split_mfma(float2* b, const float2* twx, const float2* twy, int B, int Ax,
                                                  int Bx, const PlaneGeo& g) {
  const SmallDiv dB = small_div(B), dnp = small_div(g.np), dax = small_div(Ax);
  const int n = mul24(mul24((g.h >> 1) + 1, g.np), B);
  struct Ctx {
    const float2 *z, *zc;  // Z[k], Z[h-k] of row j2 (of the lane's own column k)
    float2* out;           // null: nothing to store
    float2 w;
    int j2;
  };
  mfma_dft16_cols<-1, PREC>(
      32 * ((n + 15) >> 4),
      [&](int u) {
        const int v = (u >> 5) * 16 + (u & 15);
        const bool live = v < n, second = (u & 16) != 0;
        const int t = sdiv(live ? v : 0, dB);
        const int j2 = (live ? v : 0) - mul24(t, B);
        const int k = sdiv(t, dnp);
        const int r = mul24(t - mul24(k, g.np), g.ny) + j2;
        const int c = g.h - k;
        const int qk = sdiv(k, dax), qc = sdiv(c, dax);
        float2* pk = b + (mul24(mul24(k - mul24(qk, Ax), Bx) + qk, g.LX) + r);
        float2* pc = b + (mul24(k == 0 ? g.h : mul24(c - mul24(qc, Ax), Bx) + qc, g.LX) + r);
        float2* pz = k == 0 ? pk : pc;
        Ctx x;
        x.z = pk;
        x.zc = pz;
        x.out = live && !(second && c == k) ? (second ? pc : pk) : nullptr;
        x.w = twx[k];
        x.j2 = second ? -1 - j2 : j2;  // sign: which column of the pair
        return x;
      },
      [&](const Ctx& x, int m) {
        const float2 zk = x.z[mul24(m, B)], zc = cconj(x.zc[mul24(m, B)]);
        const float2 E = cscale(cadd(zk, zc), 0.5f);
        const float2 D = csub(zk, zc);
        const float2 T = cmul(x.w, make_float2(0.5f * D.y, -0.5f * D.x));
        return x.j2 < 0 ? cconj(csub(E, T)) : cadd(E, T);
      },
      [&](const Ctx& x, int q, float2 y) {
        if (x.out) x.out[mul24(q, B)] = q == 0 ? y : cmul(y, twy[mul24(q, x.j2 < 0 ? -1 - x.j2 : x.j2)]);
      },
      threadIdx.x, NT);
}

// the same for odd nx: units (column k, plane, j2), into the column buffer
template <int PREC, int NT>
__device__ __forceinline__ void pl_fwd_pair_mfma(const float2* b, float2* d, const float2* twy, int B, int Ax, int Bx,
                                                 const PlaneGeo& g) {
  const SmallDiv dB = small_div(B), dnp = small_div(g.np), dax = small_div(Ax);
  const int hyl = (g.ny + 1) >> 1;
  struct Ctx {
    const float2 *z, *zc;
    float2* out;
    int j2;
  };
  mfma_dft16_cols<-1, PREC>(
      mul24(mul24(g.hx, g.np), B),
      [&](int u) {
        const int t = sdiv(u, dB);
        const int j2 = u - mul24(t, B);
        const int k = sdiv(t, dnp);
        const int pl = t - mul24(k, g.np);
        const int c = k == 0 ? 0 : g.nx - k;
        const int qk = sdiv(k, dax), qc = sdiv(c, dax);
        return Ctx{b + (mul24(mul24(k - mul24(qk, Ax), Bx) + qk, g.LX) + mul24(pl, hyl)),
                   b + (mul24(mul24(c - mul24(qc, Ax), Bx) + qc, g.LX) + mul24(pl, hyl)),
                   d + (mul24(k, g.LY) + mul24(pl, g.ny) + j2), j2};
      },
      [&](const Ctx& x, int m) {
        const int y = x.j2 + mul24(m, B);
        const float2 zk = x.z[y >> 1], zc = cconj(x.zc[y >> 1]);
        const float2 D = csub(zk, zc);
        return (y & 1) ? make_float2(0.5f * D.y, -0.5f * D.x) : cscale(cadd(zk, zc), 0.5f);
      },
      [&](const Ctx& x, int q, float2 y) { x.out[mul24(q, B)] = q == 0 ? y : cmul(y, twy[mul24(q, x.j2)]); },
      threadIdx.x, NT);
}

// pass 4: unit (k1, plane, column k), columns fastest: DFT_B over the row
// positions k1 B + j2, Y[k1 + A k2] stored to the half-spectrum planes
// (column k at slot (k mod Ax) Bx + k / Ax; Ax = 1: at k).  Written through the
// L2: 144^3 12.5 -> 11.6 us, 160^3 14.3 -> 13.2 (batched launches: no change;
// the inverse's real rows, shorter runs, lose by it).
template <int B, int NT>
__device__ __forceinline__ void pl_fwd_store(const float2* b, float2* __restrict__ dst, int A, int Ax, int Bx,
                                             const PlaneGeo& g, long long pz) {
  const SmallDiv dhx = small_div(g.hx), dnc = small_div(mul24(g.np, g.hx)), dax = small_div(Ax);
  const int ncol = mul24(g.np, g.hx);
  for (int u = threadIdx.x; u < A * ncol; u += NT) {
    const int k1 = sdiv(u, dnc);
    const int c = u - mul24(k1, ncol);
    const int pl = sdiv(c, dhx);
    const int k = c - mul24(pl, g.hx);
    const int q = sdiv(k, dax);
    const int slot = (Ax > 1 && k == g.h) ? g.h : mul24(k - mul24(q, Ax), Bx) + q;
    const float2* p = b + (mul24(slot, g.LY) + mul24(pl, g.ny) + mul24(k1, B));
    float2 x[B];
#pragma unroll
    for (int j = 0; j < B; j++) x[j] = p[j];
    DftN<B, -1>::run(x);
    float2* o = dst + ((size_t)pl * (size_t)pz + (mul24(k1, g.hx) + k));
    const int st = mul24(A, g.hx);
#pragma unroll
    for (int j = 0; j < B; j++) store_through(&o[mul24(j, st)], x[j]);
  }
}

template <int NT, bool SPLIT>
__device__ __forceinline__ void plane4_fwd_body(const float* __restrict__ grid, float2* __restrict__ cg, int nx,
                                                int ny, const AxisArgs& axx, const AxisArgs& axy, int z, int np,
                                                float2* sm) {
  const PlaneGeo g = plane_geo(nx, ny, np);
  float2* twx = sm;
  float2* twy = twx + nx;
  float2* b = twy + ny;
  for (int i = threadIdx.x; i < nx; i += NT) twx[i] = axx.tw[i];
  for (int i = threadIdx.x; i < ny; i += NT) twy[i] = axy.tw[i];
  const int Ax = axx.rp.f4a, Bx = axx.rp.f4b;
  const int Ay = axy.rp.f4a, By = axy.rp.f4b;  // SPLIT: Ay = 16
  const float* src = grid + (size_t)z * nx * ny;
#define PME_CALL(L) \
  case L: pl_fwd_load<L, NT>(src, b, twx, axx.rp.tstride, Bx, g); break;
  PME_PL_SWITCH(Ax, PME_CALL)
#undef PME_CALL
  __syncthreads();
#define PME_CALL(L) \
  case L: pl_dft_b<L, -1, NT>(b, Ax, g.nxl, g.LX); break;
  PME_PL_SWITCH(Bx, PME_CALL)
#undef PME_CALL
  __syncthreads();
  float2* d = g.odd ? b + g.bx : b;
  if constexpr (SPLIT) {
    if (g.odd) {
      if (axy.prec == PREC_BF16X3)
        pl_fwd_pair_mfma<PREC_BF16X3, NT>(b, d, twy, By, Ax, Bx, g);
      else
        pl_fwd_pair_mfma<PREC_FP16X3, NT>(b, d, twy, By, Ax, Bx, g);
    } else {
      if (axy.prec == PREC_BF16X3)
        pl_fwd_split_mfma<PREC_BF16X3, NT>(b, twx, twy, By, Ax, Bx, g);
      else
        pl_fwd_split_mfma<PREC_FP16X3, NT>(b, twx, twy, By, Ax, Bx, g);
    }
  } else if (!g.odd) {
#define PME_CALL(L) \
  case L: pl_fwd_split<L, NT>(b, twx, twy, By, Ax, Bx, g); break;
    PME_PL_PAIR_SWITCH(Ay, PME_CALL)
#undef PME_CALL
  } else {
#define PME_CALL(L) \
  case L: pl_fwd_pair<L, NT>(b, d, twy, By, Ax, Bx, g); break;
    PME_PL_PAIR_SWITCH(Ay, PME_CALL)
#undef PME_CALL
  }
  __syncthreads();
  const long long pz = spec_pitch(g.hx, ny);
  float2* dst = cg + (size_t)z * (size_t)pz;
#define PME_CALL(L) \
  case L: pl_fwd_store<L, NT>(d, dst, Ay, g.odd ? 1 : Ax, g.odd ? 1 : Bx, g, pz); break;
  PME_PL_SWITCH(By, PME_CALL)
#undef PME_CALL
}

// ---- inverse ---------------------------------------------------------------------
// The factors swap roles (A the larger) so that pass 2, which holds two columns
// in registers, runs the smaller DFT, and pass 4 stores longer runs.

// pass 1: unit (j2, plane, column), columns fastest: rows j2 + B j1 from HBM
template <int A, int NT>
__device__ __forceinline__ void pl_inv_load(const float2* __restrict__ src, float2* b, const float2* tw, int B,
                                            const PlaneGeo& g, long long pz) {
  const int ncol = mul24(g.np, g.hx);
  const SmallDiv dnc = small_div(ncol), dhx = small_div(g.hx);
  const int n = B * ncol;
  const int st = mul24(B, g.hx);
  for (int u0 = 0; u0 < n; u0 += NT) {
    const int u = u0 + (int)threadIdx.x;
    const int j2 = sdiv(u, dnc);
    const int c = u - mul24(j2, ncol);
    const int pl = sdiv(c, dhx);
    const int k = c - mul24(pl, g.hx);
    const bool live = u < n;
    const float2* s = src + ((size_t)pl * (size_t)pz + (mul24(j2, g.hx) + k));
    float2 x[A];
#pragma unroll
    for (int j = 0; j < A; j++) x[j] = live ? s[mul24(j, st)] : make_float2(0.f, 0.f);
    if (u0 == 0) __syncthreads();  // twiddles in LDS (uniform branch)
    if (live) {
      DftN<A, 1>::run(x);
      float2* p = b + (mul24(k, g.LY) + mul24(pl, g.ny) + j2);
      p[0] = x[0];
#pragma unroll
      for (int q = 1; q < A; q++) p[mul24(q, B)] = cmulc(x[q], tw[mul24(q, j2)]);
    }
  }
}

// pass 1 with the DFT_16 as hi-lo products on the matrix cores: units (j2,
// plane, column), 32 of them per wave
template <int PREC, int NT>
__device__ __forceinline__ void pl_inv_load_split(const float2* __restrict__ src, float2* b, const float2* tw, int B,
                                                  const PlaneGeo& g, long long pz) {
  const int ncol = mul24(g.np, g.hx);
  const SmallDiv dnc = small_div(ncol), dhx = small_div(g.hx);
  const int st = mul24(B, g.hx);
  struct Ctx {
    const float2* s;
    float2* p;
    int j2;
  };
  __syncthreads();  // twiddles in LDS
  mfma_dft16_cols<1, PREC>(
      B * ncol,
      [&](int u) {
        const int j2 = sdiv(u, dnc);
        const int c = u - mul24(j2, ncol);
        const int pl = sdiv(c, dhx);
        const int k = c - mul24(pl, g.hx);
        return Ctx{src + ((size_t)pl * (size_t)pz + (mul24(j2, g.hx) + k)),
                   b + (mul24(k, g.LY) + mul24(pl, g.ny) + j2), j2};
      },
      [&](const Ctx& x, int m) { return x.s[mul24(m, st)]; },
      [&](const Ctx& x, int q, float2 y) { x.p[mul24(q, B)] = q == 0 ? y : cmulc(y, tw[mul24(q, x.j2)]); },
      threadIdx.x, NT);
}

// pass 2, even nx: unit (pair k <= h/2, plane, k1), k1 fastest: DFT_B of
// columns k and h-k over the positions k1 B + j2, which leaves rows k1 + A k2
// of both, then the C2R merge
//   Z[k] = P + iQ, Z[h-k] = conj(P - iQ), P = X[k] + X*[h-k], Q = w^{-k} (X[k] - X*[h-k]);
// row k1 + A k2 stays at position k1 B + k2.
template <int B, int NT>
__device__ __forceinline__ void pl_inv_merge(float2* b, const float2* twx, int A, const PlaneGeo& g) {
  const SmallDiv dA = small_div(A), dnp = small_div(g.np);
  const int n = mul24(mul24((g.h >> 1) + 1, g.np), A);
  for (int u = threadIdx.x; u < n; u += NT) {
    const int t = sdiv(u, dA);
    const int k1 = u - mul24(t, A);
    const int k = sdiv(t, dnp);
    const int r = mul24(t - mul24(k, g.np), g.ny) + mul24(k1, B);
    const int c = g.h - k;
    float2* pk = b + (mul24(k, g.LY) + r);
    float2* pc = b + (mul24(c, g.LY) + r);
    const float2 w = twx[k];
    float2 xk[B], xc[B];
#pragma unroll
    for (int j = 0; j < B; j++) {
      xk[j] = pk[j];
      xc[j] = pc[j];
    }
    DftN<B, 1>::run(xk);
    DftN<B, 1>::run(xc);
#pragma unroll
    for (int j = 0; j < B; j++) {
      const float2 v = cconj(xc[j]);
      const float2 P = cadd(xk[j], v);
      const float2 Q = cmulc(csub(xk[j], v), w);
      pk[j] = make_float2(P.x - Q.y, P.y + Q.x);
      if (c != k && k != 0) pc[j] = make_float2(P.x + Q.y, Q.x - P.y);
    }
  }
}

// pass 2, odd nx: unit (column, plane, k1), k1 fastest: DFT_B of the column
// over the positions k1 B + j2, in place
template <int B, int NT>
__device__ __forceinline__ void pl_inv_cols(float2* d, int A, const PlaneGeo& g) {
  const SmallDiv dA = small_div(A), dnp = small_div(g.np);
  const int n = mul24(mul24(g.hx, g.np), A);
  for (int u = threadIdx.x; u < n; u += NT) {
    const int t = sdiv(u, dA);
    const int k1 = u - mul24(t, A);
    const int k = sdiv(t, dnp);
    float2* p = d + (mul24(k, g.LY) + mul24(t - mul24(k, g.np), g.ny) + mul24(k1, B));
    float2 x[B];
#pragma unroll
    for (int j = 0; j < B; j++) x[j] = p[j];
    DftN<B, 1>::run(x);
#pragma unroll
    for (int j = 0; j < B; j++) p[j] = x[j];
  }
}

// pass 3, odd nx: unit (j2, x line): line Z = A + iB of the full Hermitian
// spectra of rows 2j and 2j+1 (zero past the last row) at the points j2 + Bx
// j1, DFT_A and the twiddle into the x-line buffer.  Row y sits at position
// (y mod Ay) By + y / Ay of its column.
template <int A, int NT>
__device__ __forceinline__ void pl_inv_pair(const float2* d, float2* b, const float2* tw, int tstride, int B, int Ay,
                                            int By, const PlaneGeo& g) {
  const int hyl = (g.ny + 1) >> 1;
  const SmallDiv dl = small_div(g.nxl), dh = small_div(hyl), day = small_div(Ay);
  const int BLS = mul24(B, g.LX);
  for (int u = threadIdx.x; u < B * g.nxl; u += NT) {
    const int j2 = sdiv(u, dl);
    const int l = u - mul24(j2, g.nxl);
    const int pl = sdiv(l, dh);
    const int ya = 2 * (l - mul24(pl, hyl)), yb = ya + 1;
    const bool two = yb < g.ny;
    const int qa = sdiv(ya, day), qb = sdiv(yb, day);
    const int ra = mul24(pl, g.ny) + mul24(ya - mul24(qa, Ay), By) + qa;
    const int rb = two ? mul24(pl, g.ny) + mul24(yb - mul24(qb, Ay), By) + qb : ra;
    float2 x[A];
#pragma unroll
    for (int j = 0; j < A; j++) {
      const int k = j2 + mul24(j, B);
      const bool lo = k < g.hx;
      const float2* col = d + mul24(lo ? k : g.nx - k, g.LY);
      float2 a = col[ra], v = col[rb];
      if (!two) v = make_float2(0.f, 0.f);
      if (!lo) {
        a = cconj(a);
        v = cconj(v);
      }
      x[j] = make_float2(a.x - v.y, a.y + v.x);
    }
    DftN<A, 1>::run(x);
    float2* p = b + (mul24(j2, g.LX) + l);
    const int ts = mul24(j2, tstride);
    p[0] = x[0];
#pragma unroll
    for (int q = 1; q < A; q++) p[mul24(q, BLS)] = cmulc(x[q], tw[mul24(q, ts)]);
  }
}

// pass 4: unit (x line, k1), k1 fastest (runs of A points of a row): DFT_B
// over the points j2 + B k1, x[k1 + A k2] stored to the real rows
template <int B, int NT>
__device__ __forceinline__ void pl_inv_store(const float2* b, float* __restrict__ dst, int A, int Ay, int By,
                                             const PlaneGeo& g) {
  const SmallDiv dA = small_div(A), dny = small_div(g.ny), dby = small_div(By);
  const int hyl = (g.ny + 1) >> 1;
  const SmallDiv dh = small_div(hyl);
  for (int u = threadIdx.x; u < g.nxl * A; u += NT) {
    const int l = sdiv(u, dA);
    const int k1 = u - mul24(l, A);
    const float2* p = b + (mul24(mul24(k1, B), g.LX) + l);
    float2 x[B];
#pragma unroll
    for (int j = 0; j < B; j++) x[j] = p[mul24(j, g.LX)];
    DftN<B, 1>::run(x);
    if (!g.odd) {
      const int pl = sdiv(l, dny);
      const int q = l - mul24(pl, g.ny);
      const int t = sdiv(q, dby);
      const int row = mul24(pl, g.ny) + t + mul24(Ay, q - mul24(t, By));
      float2* o = reinterpret_cast<float2*>(dst) + (mul24(row, g.h) + k1);
#pragma unroll
      for (int j = 0; j < B; j++) o[mul24(j, A)] = x[j];
    } else {
      const int pl = sdiv(l, dh);
      const int y = 2 * (l - mul24(pl, hyl));
      float* o = dst + (mul24(mul24(pl, g.ny) + y, g.nx) + k1);
#pragma unroll
      for (int j = 0; j < B; j++) o[mul24(j, A)] = x[j].x;
      if (y + 1 < g.ny) {
#pragma unroll
        for (int j = 0; j < B; j++) o[mul24(j, A) + g.nx] = x[j].y;
      }
    }
  }
}

template <int NT, bool SPLIT>
__device__ __forceinline__ void plane4_inv_body(const float2* __restrict__ cg, float* __restrict__ grid, int nx,
                                                int ny, const AxisArgs& axx, const AxisArgs& axy, int z, int np,
                                                float2* sm) {
  const PlaneGeo g = plane_geo(nx, ny, np);
  float2* twx = sm;
  float2* twy = twx + nx;
  float2* b = twy + ny;
  for (int i = threadIdx.x; i < nx; i += NT) twx[i] = axx.tw[i];
  for (int i = threadIdx.x; i < ny; i += NT) twy[i] = axy.tw[i];
  const int Ax = axx.rp.f4b, Bx = axx.rp.f4a;
  const int Ay = SPLIT ? 16 : axy.rp.f4b, By = SPLIT ? axy.rp.f4b : axy.rp.f4a;
  const long long pz = spec_pitch(g.hx, ny);
  const float2* src = cg + (size_t)z * (size_t)pz;
  float2* d = g.odd ? b + g.bx : b;  // columns
  if constexpr (SPLIT) {
    if (axy.prec == PREC_BF16X3)
      pl_inv_load_split<PREC_BF16X3, NT>(src, d, twy, By, g, pz);
    else
      pl_inv_load_split<PREC_FP16X3, NT>(src, d, twy, By, g, pz);
  } else {
#define PME_CALL(L) \
  case L: pl_inv_load<L, NT>(src, d, twy, By, g, pz); break;
    PME_PL_SWITCH(Ay, PME_CALL)
#undef PME_CALL
  }
  __syncthreads();
  if (!g.odd) {
#define PME_CALL(L) \
  case L: pl_inv_merge<L, NT>(b, twx, Ay, g); break;
    PME_PL_PAIR_SWITCH(By, PME_CALL)
#undef PME_CALL
    __syncthreads();
#define PME_CALL(L) \
  case L: pl_dft_a<L, 1, NT>(b, twx, axx.rp.tstride, Bx, g.nxl, g.LX); break;
    PME_PL_SWITCH(Ax, PME_CALL)
#undef PME_CALL
  } else {
#define PME_CALL(L) \
  case L: pl_inv_cols<L, NT>(d, Ay, g); break;
    PME_PL_PAIR_SWITCH(By, PME_CALL)
#undef PME_CALL
    __syncthreads();
#define PME_CALL(L) \
  case L: pl_inv_pair<L, NT>(d, b, twx, axx.rp.tstride, Bx, Ay, By, g); break;
    PME_PL_SWITCH(Ax, PME_CALL)
#undef PME_CALL
  }
  __syncthreads();
  float* dst = grid + (size_t)z * nx * ny;
#define PME_CALL(L) \
  case L: pl_inv_store<L, NT>(b, dst, Ax, Ay, By, g); break;
  PME_PL_SWITCH(Bx, PME_CALL)
#undef PME_CALL
}

// ---- kernels -----------------------------------------------------------------------

template <int NT, bool SPLIT>
__global__ __launch_bounds__(NT, 4) void k_plane4_fwd(const float* __restrict__ grid, float2* __restrict__ cg, int nx,
                                                      int ny, AxisArgs axx, AxisArgs axy) {
  extern __shared__ __align__(16) float2 sm[];
  plane4_fwd_body<NT, SPLIT>(grid, cg, nx, ny, axx, axy, blockIdx.x, 1, sm);
}

// With a pending energy/virial reduction the launch has one more workgroup
// that performs it alone, so no plane's workgroup waits for it.
template <int NT, bool SPLIT>
__global__ __launch_bounds__(NT, 4) void k_plane4_inv(const float2* __restrict__ cg, float* __restrict__ grid, int nx,
                                                      int ny, int nz, AxisArgs axx, AxisArgs axy, EvReduce red) {
  extern __shared__ __align__(16) float2 sm[];
  if ((int)blockIdx.x >= nz) {
    ev_reduce_block<NT>(red);
    return;
  }
  plane4_inv_body<NT, SPLIT>(cg, grid, nx, ny, axx, axy, blockIdx.x, 1, sm);
}

// Threads of a single-system plane workgroup: one unit of work each in the
// widest pass, as far as that goes.
static int plane4_threads(int nx, int ny, const AxisArgs& ax, const AxisArgs& ay) {
  const PlaneGeo g = plane_geo(nx, ny, 1);
  const int u = std::max(g.nxl * ax.rp.f4b, g.hx * ay.rp.f4b);
  return u <= 256 ? 256 : (u <= 512 ? 512 : 1024);
}

template <bool SPLIT>
static void plane4_fwd_as(const float* grid, float2* cg, int nx, int ny, int nz, const AxisArgs& ax,
                          const AxisArgs& ay, size_t lds, hipStream_t s) {
  switch (plane4_threads(nx, ny, ax, ay)) {
    case 256: hipLaunchKernelGGL((k_plane4_fwd<256, SPLIT>), dim3(nz), dim3(256), lds, s, grid, cg, nx, ny, ax, ay); break;
    case 512: hipLaunchKernelGGL((k_plane4_fwd<512, SPLIT>), dim3(nz), dim3(512), lds, s, grid, cg, nx, ny, ax, ay); break;
    default: hipLaunchKernelGGL((k_plane4_fwd<1024, SPLIT>), dim3(nz), dim3(1024), lds, s, grid, cg, nx, ny, ax, ay); break;
  }
}

hipError_t launch_plane4_fwd(const float* grid, float2* cg, int nx, int ny, int nz, const AxisArgs& ax,
                             const AxisArgs& ay, hipStream_t s) {
  const size_t lds = fft_plane4_lds_bytes(nx, ny, 1);
  const PlaneKind kind = plane_kind(nx, ny, ax.rp, ay.rp, ay.prec);
  if (kind == PLANE_FOUR_STEP)
    plane4_fwd_as<false>(grid, cg, nx, ny, nz, ax, ay, lds, s);
  else if (kind == PLANE_FOUR_STEP_SPLIT)
    plane4_fwd_as<true>(grid, cg, nx, ny, nz, ax, ay, lds, s);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

template <bool SPLIT>
static void plane4_inv_as(const float2* cg, float* grid, int nx, int ny, int nz, const AxisArgs& ax,
                          const AxisArgs& ay, const EvReduce& red, size_t lds, hipStream_t s) {
  const dim3 gr(nz + ((red.nsolve > 0 || red.nself > 0) ? 1 : 0));
  switch (plane4_threads(nx, ny, ax, ay)) {
    case 256: hipLaunchKernelGGL((k_plane4_inv<256, SPLIT>), gr, dim3(256), lds, s, cg, grid, nx, ny, nz, ax, ay, red); break;
    case 512: hipLaunchKernelGGL((k_plane4_inv<512, SPLIT>), gr, dim3(512), lds, s, cg, grid, nx, ny, nz, ax, ay, red); break;
    default: hipLaunchKernelGGL((k_plane4_inv<1024, SPLIT>), gr, dim3(1024), lds, s, cg, grid, nx, ny, nz, ax, ay, red); break;
  }
}

hipError_t launch_plane4_inv(const float2* cg, float* grid, int nx, int ny, int nz, const AxisArgs& ax,
                             const AxisArgs& ay, const EvReduce& red, hipStream_t s) {
  const size_t lds = fft_plane4_lds_bytes(nx, ny, 1);
  const PlaneKind kind = plane_kind(nx, ny, ax.rp, ay.rp, ay.prec);
  if (kind == PLANE_FOUR_STEP)
    plane4_inv_as<false>(cg, grid, nx, ny, nz, ax, ay, red, lds, s);
  else if (kind == PLANE_FOUR_STEP_SPLIT)
    plane4_inv_as<true>(cg, grid, nx, ny, nz, ax, ay, red, lds, s);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

// Batched: items are (system, first plane), plane4_group planes each (fewer at
// the top of the grid); NT = kPlaneBlock / 2 for systems whose plane fits half
// the LDS budget, two workgroups per CU.  Held to 128 VGPRs (four waves per SIMD),
// where the inverse spills one VGPR in FP32 and three in split precision.
template <int INV, int NT, bool SPLIT>
__global__ __launch_bounds__(NT, 4) void k_batch_plane4(const SysDesc* __restrict__ sys,
                                                        const WorkItem* __restrict__ items, int nitems, int reduce,
                                                        int maxnp) {
  extern __shared__ __align__(16) float2 sm[];
  for (int it = blockIdx.x; it < nitems; it += gridDim.x) {
    const WorkItem w = uniform_item(items[it]);
    const SysDesc& d = sys[w.sys];
    const int np = min(plane4_group(d.bin.nx, d.bin.ny, maxnp, NT < kPlaneBlock), d.bin.nz - w.idx);
    if (INV) {
      if (reduce && w.idx == 0 && (d.sa.calc_ev || d.calc_self)) batch_ev_reduce<NT>(d);
      plane4_inv_body<NT, SPLIT>(d.cgrid, d.grid, d.bin.nx, d.bin.ny, d.ax[0], d.ax[1], w.idx, np, sm);
    } else {
      plane4_fwd_body<NT, SPLIT>(d.grid, d.cgrid, d.bin.nx, d.bin.ny, d.ax[0], d.ax[1], w.idx, np, sm);
    }
    __syncthreads();
  }
}

template <bool SPLIT>
static void batch_plane4_as(int inverse, int reduce, int maxnp, int half, const SysDesc* sys, const WorkItem* items,
                            int nitems, int grid, size_t lds, hipStream_t s) {
  constexpr int F = kPlaneBlock, H = kPlaneBlock / 2;
  if (inverse && half)
    hipLaunchKernelGGL((k_batch_plane4<1, H, SPLIT>), dim3(grid), dim3(H), lds, s, sys, items, nitems, reduce, maxnp);
  else if (inverse)
    hipLaunchKernelGGL((k_batch_plane4<1, F, SPLIT>), dim3(grid), dim3(F), lds, s, sys, items, nitems, reduce, maxnp);
  else if (half)
    hipLaunchKernelGGL((k_batch_plane4<0, H, SPLIT>), dim3(grid), dim3(H), lds, s, sys, items, nitems, reduce, maxnp);
  else
    hipLaunchKernelGGL((k_batch_plane4<0, F, SPLIT>), dim3(grid), dim3(F), lds, s, sys, items, nitems, reduce, maxnp);
}

hipError_t launch_batch_plane4(int inverse, int reduce, int maxnp, int split, int half, const SysDesc* sys,
                               const WorkItem* items, int nitems, int grid, size_t lds, hipStream_t s) {
  if (nitems <= 0) return hipSuccess;
  if (maxnp < 1 || maxnp > kPlaneGroupMax) return hipErrorInvalidValue;
  if (split)
    batch_plane4_as<true>(inverse, reduce, maxnp, half, sys, items, nitems, grid, lds, s);
  else
    batch_plane4_as<false>(inverse, reduce, maxnp, half, sys, items, nitems, grid, lds, s);
  return hipGetLastError();
}

}  // namespace pme
