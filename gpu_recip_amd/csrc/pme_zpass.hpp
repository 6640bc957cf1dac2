// pme_zpass.hpp -- device code of the reciprocal convolution (influence
// function, energy and virial) and of the fused z pass as a register four-step
// FFT, shared by the kernels of pme_fft.hip and pme_zsolve.hip.
#pragma once
#include "pme_internal.hpp"

namespace pme {

// ------------------------------------------------------- influence function --

// eterm at (k1, k2, k3) and the energy/virial terms of that point,
// scalar_sum_ortho_kernel CudaPMERecip.cu:671-704
__device__ __forceinline__ float eterm_at(const SolveArgs& s, int k1, int k2, int k3, float& mh1, float& mh2,
                                          float& mh3, float& msq_inv) {
  const int m1 = k1 >= s.nf1 ? k1 - s.n1 : k1;
  const int m2 = k2 >= s.nf2 ? k2 - s.n2 : k2;
  const int m3 = k3 >= s.nf3 ? k3 - s.n3 : k3;
  mh1 = s.r1 * (float)m1;
  mh2 = s.r2 * (float)m2;
  mh3 = s.r3 * (float)m3;
  // grouped as in solve_lines, which takes the (k1, k2) factors out of its
  // loop over k3, so both give the same value; the fused multiply-adds are
  // explicit so that every kernel rounds them alike
  const float s12 = fmaf(mh2, mh2, mh1 * mh1);
  const float msq = fmaf(mh3, mh3, s12);
  const float p12 = s.piv_inv * s.pf1[k1] * s.pf2[k2];
  // hardware reciprocal and exponential (1-2 ulp), as the reference's fast-math build
  msq_inv = __builtin_amdgcn_rcpf(msq);
  return __expf(-s.fac * msq) * p12 * s.pf3[k3] * msq_inv;
}

// Multiply one half-spectrum point by eterm; accumulate energy/virial with
// the reference's weights (mirror term for every k1 >= 1, :708-741).  The
// mirror point (n1-k1, -k2, -k3) has the same |m|^2 and, bsp_mod being
// symmetric, the same eterm; its m components are -m except on a Nyquist
// plane of an even axis (m = -n/2 maps to itself), so the diagonal terms
// double and each off-diagonal term m_a m_b doubles or cancels.
__device__ __forceinline__ float2 solve_point(const SolveArgs& s, float2 q, int k1, int k2, int k3, double* acc) {
  if ((k1 | k2 | k3) == 0) return make_float2(0.f, 0.f);
  float mh1, mh2, mh3, msq_inv;
  const float eterm = eterm_at(s, k1, k2, k3, mh1, mh2, mh3, msq_inv);
  if (s.calc_ev) {
    const float q2 = fmaf(q.y, q.y, q.x * q.x);
    const float tmp1 = eterm * q2;
    const float vterm = 2.0f * (s.fac + msq_inv);
    const float tmp2 = tmp1 * vterm;
    // weight of the point (1) plus its mirror (1 when k1 >= 1)
    const double w = k1 >= 1 ? 2.0 : 1.0;
    // mirror sign of each m component: +1 when it maps to itself
    const bool f1 = !(2 * k1 == s.n1), f2 = !(2 * k2 == s.n2 || k2 == 0), f3 = !(2 * k3 == s.n3 || k3 == 0);
    const double w12 = k1 >= 1 ? (f1 == f2 ? 2.0 : 0.0) : 1.0;
    const double w13 = k1 >= 1 ? (f1 == f3 ? 2.0 : 0.0) : 1.0;
    const double w23 = k1 >= 1 ? (f2 == f3 ? 2.0 : 0.0) : 1.0;
    acc[0] += w * (double)tmp1;
    acc[1] += w * (double)(tmp1 * (vterm * mh1 * mh1 - 1.0f));
    acc[2] += w12 * (double)(tmp2 * mh1 * mh2);
    acc[3] += w13 * (double)(tmp2 * mh1 * mh3);
    acc[4] += w * (double)(tmp1 * (vterm * mh2 * mh2 - 1.0f));
    acc[5] += w23 * (double)(tmp2 * mh2 * mh3);
    acc[6] += w * (double)(tmp1 * (vterm * mh3 * mh3 - 1.0f));
  }
  return cscale(q, eterm);
}

// eterm of a triclinic box at mapped wave numbers (m1, m2, m3), k3 = its z
// index: m-hat = m1 R[0][:] + m2 R[1][:] + m3 R[2][:] (rows of recip).
__device__ __forceinline__ float eterm_tric(const SolveArgs& s, int k1, int k2, int k3, int m1, int m2, int m3,
                                            float* mh, float& msq_inv) {
  const float f1 = (float)m1, f2 = (float)m2, f3 = (float)m3;
  mh[0] = fmaf(s.rt[6], f3, fmaf(s.rt[3], f2, s.rt[0] * f1));
  mh[1] = fmaf(s.rt[7], f3, fmaf(s.rt[4], f2, s.rt[1] * f1));
  mh[2] = fmaf(s.rt[8], f3, fmaf(s.rt[5], f2, s.rt[2] * f1));
  const float msq = fmaf(mh[2], mh[2], fmaf(mh[1], mh[1], mh[0] * mh[0]));
  msq_inv = __builtin_amdgcn_rcpf(msq);
  return __expf(-s.fac * msq) * (s.piv_inv * s.pf1[k1] * s.pf2[k2]) * s.pf3[k3] * msq_inv;
}

// energy and virial terms of one point (weight 1), the order of acc as in solve_point
__device__ __forceinline__ void ev_terms(const SolveArgs& s, float eterm, float q2, const float* mh, float msq_inv,
                                         double* acc) {
  const float tmp1 = eterm * q2;
  const float vterm = 2.0f * (s.fac + msq_inv);
  const float tmp2 = tmp1 * vterm;
  acc[0] += (double)tmp1;
  acc[1] += (double)(tmp1 * (vterm * mh[0] * mh[0] - 1.0f));
  acc[2] += (double)(tmp2 * mh[0] * mh[1]);
  acc[3] += (double)(tmp2 * mh[0] * mh[2]);
  acc[4] += (double)(tmp1 * (vterm * mh[1] * mh[1] - 1.0f));
  acc[5] += (double)(tmp2 * mh[1] * mh[2]);
  acc[6] += (double)(tmp1 * (vterm * mh[2] * mh[2] - 1.0f));
}

// solve_point for a triclinic box: the same weights (the point, plus its
// mirror (n1-k1, -k2, -k3) for every k1 >= 1), but the mirror's m-hat is not
// minus the point's on a Nyquist plane, so its eterm and virial terms are
// evaluated from its own wave numbers.
__device__ __forceinline__ float2 solve_point_tric(const SolveArgs& s, float2 q, int k1, int k2, int k3, double* acc) {
  if ((k1 | k2 | k3) == 0) return make_float2(0.f, 0.f);
  const int m1 = k1 >= s.nf1 ? k1 - s.n1 : k1;
  const int m2 = k2 >= s.nf2 ? k2 - s.n2 : k2;
  const int m3 = k3 >= s.nf3 ? k3 - s.n3 : k3;
  float mh[3], msq_inv;
  const float eterm = eterm_tric(s, k1, k2, k3, m1, m2, m3, mh, msq_inv);
  if (s.calc_ev) {
    const float q2 = fmaf(q.y, q.y, q.x * q.x);
    ev_terms(s, eterm, q2, mh, msq_inv, acc);
    if (k1 >= 1) {
      const int k1s = s.n1 - k1, k2s = k2 ? s.n2 - k2 : 0, k3s = k3 ? s.n3 - k3 : 0;
      const int m1s = k1s >= s.nf1 ? k1s - s.n1 : k1s;
      const int m2s = k2s >= s.nf2 ? k2s - s.n2 : k2s;
      const int m3s = k3s >= s.nf3 ? k3s - s.n3 : k3s;
      float ms[3], msq_inv_s;
      const float eterm_s = eterm_tric(s, k1s, k2s, k3s, m1s, m2s, m3s, ms, msq_inv_s);
      ev_terms(s, eterm_s, q2, ms, msq_inv_s, acc);
    }
  }
  return cscale(q, eterm);
}

// The influence function over the z lines of a column tile (in LDS, point j
// of line l at res[j * TX + l]; lines l < nl are kx = kx0 + l at ky = k2).
// Thread t owns line t mod TX and visits k3 = t / TX, t / TX + kBlock / TX,
// ..., so the (k1, k2) factors of eterm and of the energy/virial terms are
// formed once per thread: scalar_sum_ortho_kernel CudaPMERecip.cu:671-747
// per point, with the sums over k3 of one line taken before the line's
// constant factors are applied.  Per line, with the point weight w (2 when
// k1 >= 1: the point and its mirror), tmp1 = eterm |Q|^2, tmp2 = tmp1 vterm:
//   E   += w sum tmp1                  V11 += w (mh1^2 sum tmp2 - sum tmp1)
//   V22 += w (mh2^2 sum tmp2 - sum tmp1)  V33 += w (sum tmp2 mh3^2 - sum tmp1)
//   V12 += w12 mh1 mh2 sum tmp2      V13 += mh1 sum w13 tmp2 mh3
//   V23 += mh2 sum w23 tmp2 mh3
// (the off-diagonal mirror weights are those of solve_point; w13 and w23
// depend on k3 through the zero/Nyquist test of m3).
__device__ __forceinline__ void solve_lines(const SolveArgs& s, float2* __restrict__ res, int n, int TX, int nl,
                                            int c0, int hxd, double* acc) {
  const int tid = threadIdx.x;
  const SmallDiv dtx = small_div(TX);
  const int j0 = sdiv(tid, dtx);
  const int l = tid - j0 * TX;
  const int jstep = sdiv(kBlock, dtx);  // >= 4: column tiles are at most 64 wide
  static_assert(kBlock >= 4 * 64, "solve_lines: every line needs a thread");
  if (j0 >= jstep || l >= nl) return;
  // line c0 + l of the z pass: flattened (ky, kx) of the z plane, rows of hxd
  const int c = c0 + l;
  const int k2 = sdiv(c, small_div(hxd));
  const int k1 = c - k2 * hxd;
  const int m1 = k1 >= s.nf1 ? k1 - s.n1 : k1;
  const int m2 = k2 >= s.nf2 ? k2 - s.n2 : k2;
  const float mh1 = s.r1 * (float)m1;
  const float mh2 = s.r2 * (float)m2;
  const float s12 = fmaf(mh2, mh2, mh1 * mh1);
  const float p12 = s.piv_inv * s.pf1[k1] * s.pf2[k2];
  const bool f1 = !(2 * k1 == s.n1), f2 = !(2 * k2 == s.n2 || k2 == 0);
  const bool k1pos = k1 >= 1;
  double sA = 0.0, sB = 0.0, sC = 0.0, sD13 = 0.0, sD23 = 0.0;
  for (int j = j0; j < n; j += jstep) {
    float2* pt = res + mul24(j, TX) + l;
    if ((k1 | k2 | j) == 0) {
      *pt = make_float2(0.f, 0.f);
      continue;
    }
    const int m3 = j >= s.nf3 ? j - s.n3 : j;
    const float mh3 = s.r3 * (float)m3;
    const float msq = fmaf(mh3, mh3, s12);
    const float msq_inv = __builtin_amdgcn_rcpf(msq);
    const float eterm = __expf(-s.fac * msq) * p12 * s.pf3[j] * msq_inv;
    const float2 q = *pt;
    if (s.calc_ev) {
      const float q2 = fmaf(q.y, q.y, q.x * q.x);
      const float tmp1 = eterm * q2;
      const float vterm = 2.0f * (s.fac + msq_inv);
      const float tmp2 = tmp1 * vterm;
      const float t3 = tmp2 * mh3;
      const bool f3 = !(2 * j == s.n3 || j == 0);
      const float w13 = k1pos ? (f1 == f3 ? 2.f : 0.f) : 1.f;
      const float w23 = k1pos ? (f2 == f3 ? 2.f : 0.f) : 1.f;
      sA += (double)tmp1;
      sB += (double)tmp2;
      sC += (double)(t3 * mh3);
      sD13 += (double)(w13 * t3);
      sD23 += (double)(w23 * t3);
    }
    *pt = cscale(q, eterm);
  }
  if (s.calc_ev) {
    const double w = k1pos ? 2.0 : 1.0;
    const double w12 = k1pos ? (f1 == f2 ? 2.0 : 0.0) : 1.0;
    const double a1 = (double)mh1, a2 = (double)mh2;
    acc[0] += w * sA;
    acc[1] += w * (a1 * a1 * sB - sA);
    acc[2] += w12 * a1 * a2 * sB;
    acc[3] += a1 * sD13;
    acc[4] += w * (a2 * a2 * sB - sA);
    acc[5] += a2 * sD23;
    acc[6] += w * (sC - sA);
  }
}

// Per-workgroup energy/virial partial (fixed summation order inside the
// workgroup).  The total is formed later by ev_reduce_block in one workgroup.
__device__ __forceinline__ void ev_partial(const SolveArgs& s, double* acc, double* sh, int blk) {
  block_sum<7>(acc, sh);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int c = 0; c < 7; c++) s.partial[(size_t)blk * 7 + c] = acc[c];
  }
}

// ---- z pass as a register four-step FFT -------------------------------------
// n = N1 N2, j = j2 + N2 j1, k = k1 + N1 k2:
//   X[k1 + N1 k2] = sum_j2 w_N2^{j2 k2} w_n^{j2 k1} sum_j1 w_N1^{j1 k1} x[j2 + N2 j1].
// Work unit (line l, q): in the forward half q = j2 (an N1-point DFT of the
// column j2 + N2 j1 in registers, the twiddle w_n^{j2 k1}, one LDS
// exchange), then q = k1 (an N2-point DFT in registers).  That thread then
// holds the whole line's spectrum at k3 = k1 + N1 k2, applies the influence
// function there and runs the inverse the same way back (the conjugate
// steps in reverse order).  Two LDS exchanges per direction instead of one
// per radix stage, and no index arithmetic inside the DFTs.
#define PME_F4_PAIRS(X)                                                                             \
  X(0, 4, 4) X(1, 4, 5) X(2, 4, 6) X(3, 5, 5) X(4, 3, 9) X(5, 5, 6) X(6, 4, 8) X(7, 6, 6) X(8, 5, 8) \
  X(9, 5, 9) X(10, 6, 8) X(11, 5, 10) X(12, 6, 9) X(13, 6, 10) X(14, 8, 8) X(15, 8, 9) X(16, 5, 15)  \
  X(17, 8, 10) X(18, 9, 9) X(19, 9, 10) X(20, 8, 12) X(21, 10, 10) X(22, 9, 12) X(23, 10, 12)        \
  X(24, 8, 16) X(25, 9, 15) X(26, 12, 12) X(27, 10, 15) X(28, 10, 16) X(29, 12, 15) X(30, 12, 16)
// z pass only (their longer codelet has no place among the y passes' codelets;
// 81 x 75 x 125: 61.2 -> 58.8 us per solve against Stockham stages in z)
#define PME_F4_Z_PAIRS(X) X(31, 5, 25) X(32, 9, 18)

// Register class of a factor pair.  A kernel that dispatches over several
// pairs is allocated the registers of their union, which grows well beyond
// the largest single pair (all 31 pairs and the Stockham stages: 157 VGPRs,
// three waves per SIMD; one pair: 72 to 118).  The batched z pass therefore
// has one kernel per class: class 0 holds the pairs with N2 <= 10 and 5 x 15
// (75, a common edge; held to 128 VGPRs, four waves per SIMD, with five
// spilled), class 1 the pairs up to 12 x 16 (125 VGPRs), class 2 those with a longer
// codelet (153 VGPRs, not held to 128).
constexpr int f4_class_of(int n1, int n2) {
  return (n2 <= 10 || (n1 == 5 && n2 == 15)) ? 0 : (n2 <= 16 ? 1 : 2);
}

// eterm of one point of a z line; (k1, k2) factors precomputed (as in
// solve_lines, so the value is the same)
struct LineFactors {
  float mh1, mh2, s12, p12;
  bool f1, f2, k1pos;
  int k1, k2;
};
__device__ __forceinline__ LineFactors line_factors(const SolveArgs& s, int k1, int k2) {
  LineFactors f;
  const int m1 = k1 >= s.nf1 ? k1 - s.n1 : k1;
  const int m2 = k2 >= s.nf2 ? k2 - s.n2 : k2;
  f.mh1 = s.r1 * (float)m1;
  f.mh2 = s.r2 * (float)m2;
  f.s12 = fmaf(f.mh2, f.mh2, f.mh1 * f.mh1);
  f.p12 = s.piv_inv * s.pf1[k1] * s.pf2[k2];
  f.f1 = !(2 * k1 == s.n1);
  f.f2 = !(2 * k2 == s.n2 || k2 == 0);
  f.k1pos = k1 >= 1;
  f.k1 = k1;
  f.k2 = k2;
  return f;
}

// Q <- eterm Q at k3 of the line; energy/virial sums as in solve_lines
__device__ __forceinline__ float2 solve_line_point(const SolveArgs& s, const LineFactors& f, int k3, float2 q,
                                                   double* sums) {
  if ((f.k1 | f.k2 | k3) == 0) return make_float2(0.f, 0.f);
  const int m3 = k3 >= s.nf3 ? k3 - s.n3 : k3;
  const float mh3 = s.r3 * (float)m3;
  const float msq = fmaf(mh3, mh3, f.s12);
  const float msq_inv = __builtin_amdgcn_rcpf(msq);
  const float eterm = __expf(-s.fac * msq) * f.p12 * s.pf3[k3] * msq_inv;
  if (s.calc_ev) {
    const float q2 = fmaf(q.y, q.y, q.x * q.x);
    const float tmp1 = eterm * q2;
    const float vterm = 2.0f * (s.fac + msq_inv);
    const float tmp2 = tmp1 * vterm;
    const float t3 = tmp2 * mh3;
    const bool f3 = !(2 * k3 == s.n3 || k3 == 0);
    const float w13 = f.k1pos ? (f.f1 == f3 ? 2.f : 0.f) : 1.f;
    const float w23 = f.k1pos ? (f.f2 == f3 ? 2.f : 0.f) : 1.f;
    sums[0] += (double)tmp1;
    sums[1] += (double)tmp2;
    sums[2] += (double)(t3 * mh3);
    sums[3] += (double)(w13 * t3);
    sums[4] += (double)(w23 * t3);
  }
  return cscale(q, eterm);
}

__device__ __forceinline__ void fold_line_sums(const LineFactors& f, const double* sums, double* acc) {
  const double w = f.k1pos ? 2.0 : 1.0;
  const double w12 = f.k1pos ? (f.f1 == f.f2 ? 2.0 : 0.0) : 1.0;
  const double a1 = (double)f.mh1, a2 = (double)f.mh2;
  acc[0] += w * sums[0];
  acc[1] += w * (a1 * a1 * sums[1] - sums[0]);
  acc[2] += w12 * a1 * a2 * sums[1];
  acc[3] += a1 * sums[3];
  acc[4] += w * (a2 * a2 * sums[1] - sums[0]);
  acc[5] += a2 * sums[4];
  acc[6] += w * (sums[2] - sums[0]);
}

// The same for a triclinic box: m-hat = m1 R[0][:] + m2 R[1][:] + m3 R[2][:], the
// first two terms formed once per line.  eterm is that of eterm_tric.  The
// mirror point of every k1 >= 1 has -m-hat and so the same terms, except on a
// Nyquist plane, where its terms are evaluated from its own wave numbers.
struct LineTric {
  float b[3], p12;
  bool nyq;  // the line lies on a Nyquist plane of x or y
  int k1, k2;
};
__device__ __forceinline__ LineTric line_tric(const SolveArgs& s, int k1, int k2) {
  LineTric f;
  const float f1 = (float)(k1 >= s.nf1 ? k1 - s.n1 : k1), f2 = (float)(k2 >= s.nf2 ? k2 - s.n2 : k2);
#pragma unroll
  for (int c = 0; c < 3; c++) f.b[c] = fmaf(s.rt[3 + c], f2, s.rt[c] * f1);
  f.p12 = s.piv_inv * s.pf1[k1] * s.pf2[k2];
  f.nyq = 2 * k1 == s.n1 || 2 * k2 == s.n2;
  f.k1 = k1;
  f.k2 = k2;
  return f;
}
__device__ __forceinline__ float2 solve_line_tric(const SolveArgs& s, const LineTric& f, int k3, float2 q,
                                                  double* acc) {
  if ((f.k1 | f.k2 | k3) == 0) return make_float2(0.f, 0.f);
  const float f3 = (float)(k3 >= s.nf3 ? k3 - s.n3 : k3);
  float mh[3];
#pragma unroll
  for (int c = 0; c < 3; c++) mh[c] = fmaf(s.rt[6 + c], f3, f.b[c]);
  const float msq = fmaf(mh[2], mh[2], fmaf(mh[1], mh[1], mh[0] * mh[0]));
  const float msq_inv = __builtin_amdgcn_rcpf(msq);
  const float eterm = __expf(-s.fac * msq) * f.p12 * s.pf3[k3] * msq_inv;
  if (s.calc_ev) {
    const float q2 = fmaf(q.y, q.y, q.x * q.x);
    const bool own_mirror = f.k1 >= 1 && (f.nyq || 2 * k3 == s.n3);
    ev_terms(s, eterm * ((f.k1 >= 1 && !own_mirror) ? 2.0f : 1.0f), q2, mh, msq_inv, acc);
    if (own_mirror) {
      const int k1s = s.n1 - f.k1, k2s = f.k2 ? s.n2 - f.k2 : 0, k3s = k3 ? s.n3 - k3 : 0;
      float ms[3], msq_inv_s;
      const float eterm_s =
          eterm_tric(s, k1s, k2s, k3s, k1s >= s.nf1 ? k1s - s.n1 : k1s, k2s >= s.nf2 ? k2s - s.n2 : k2s,
                     k3s >= s.nf3 ? k3s - s.n3 : k3s, ms, msq_inv_s);
      ev_terms(s, eterm_s, q2, ms, msq_inv_s, acc);
    }
  }
  return cscale(q, eterm);
}

// Influence function over the N2 points k3 = k1 + N1 k2 (X[k2]) of line `line` of
// the flattened (ky, kx), rows of hxd
template <int N1, int N2, bool TRIC>
__device__ __forceinline__ void solve_line_points(const SolveArgs& sa, float2* X, int k1, int line, int hxd,
                                                  double* acc) {
  const int ky = sdiv(line, small_div(hxd));
  if constexpr (TRIC) {
    const LineTric f = line_tric(sa, line - ky * hxd, ky);
#pragma unroll
    for (int k2 = 0; k2 < N2; k2++) X[k2] = solve_line_tric(sa, f, k1 + N1 * k2, X[k2], acc);
  } else {
    const LineFactors f = line_factors(sa, line - ky * hxd, ky);
    double sums[5] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int k2 = 0; k2 < N2; k2++) X[k2] = solve_line_point(sa, f, k1 + N1 * k2, X[k2], sums);
    if (sa.calc_ev) fold_line_sums(f, sums, acc);
  }
}

// Middle pass of the register four-step z pass: forward second half, influence
// function, inverse first half.  Unit (l, k1), in place on the N2 points (k1 N2 +
// j2) of b; lines kx0 + l of the flattened (ky, kx), rows of hxd.
template <int N1, int N2, bool TRIC>
__device__ __forceinline__ void zsolve_middle(float2* __restrict__ b, const float2* __restrict__ tw, int ts, int TX,
                                              int kx0, int nl, int hxd, const SolveArgs& sa, double* acc) {
  const int tsh = __builtin_ctz(TX);
  for (int u = threadIdx.x; u < N1 * TX; u += kBlock) {
    const int k1 = (u >> tsh);
    const int l = u - k1 * TX;
    float2 X[N2];
#pragma unroll
    for (int j2 = 0; j2 < N2; j2++) X[j2] = b[(k1 * N2 + j2) * TX + l];
    DftN<N2, -1>::run(X);  // X[k2]: point k3 = k1 + N1 k2
    if (l < nl) solve_line_points<N1, N2, TRIC>(sa, X, k1, kx0 + l, hxd, acc);
    DftN<N2, +1>::run(X);  // X[j2]
#pragma unroll
    for (int j2 = 0; j2 < N2; j2++) {
      const float2 t = tw[mul24(j2 * k1, ts)];
      const float2 z = j2 == 0 ? X[0] : cmul(X[j2], make_float2(t.x, -t.y));
      b[(k1 * N2 + j2) * TX + l] = z;
    }
  }
}

// One column tile of the z pass (as fft_cols_body<COL_FWD_SOLVE_INV>) with
// n = N1 N2: TX consecutive lines c0 .. c0+TX-1 of the flattened (ky, kx)
// index of a z plane (rows of hxd), point j of line l at base + j pt_stride
// + l.  sm: twiddles (ntw) and ONE n*TX buffer b: the first half reads its
// columns straight from HBM into registers and writes b at (k1 N2 + j2); the
// middle pass reads and rewrites the same N2 points of b per unit (in place);
// the last half reads b and stores straight to HBM.  Lanes run along l, so
// every HBM access of a wave is two runs of TX consecutive float2.  The stores
// are written through (144^3 10.9 -> 9.8 us, 160^3 17.3 -> 15.9, the 64-system
// batch 49.4 -> 48.2).  TRIC: a triclinic box's influence function.
template <int N1, int N2, bool TRIC = false>
__device__ __forceinline__ void zsolve_four_step(float2* __restrict__ cg, int hx, int TX, long long pt_stride,
                                                 long long outer_stride, const AxisArgs& ax, const SolveArgs& sa,
                                                 int tx, int ty, int blk, float2* sm, int hxd) {
  __shared__ double sh_red[7 * (kBlock / 64)];
  const int tid = threadIdx.x;
  float2* tw = sm;
  float2* b = sm + ax.ntw;
  for (int i = tid; i < ax.ntw; i += kBlock) tw[i] = ax.tw[i];
  const int ts = ax.rp.tstride;
  const int kx0 = tx * TX;
  const int nl = min(TX, hx - kx0);
  // the tile's first point (uniform) and 32-bit point offsets from it: a z
  // line spans n * pt_stride < 2^27 points (edges <= 512)
  float2* __restrict__ tile = cg + ((size_t)kx0 + (size_t)ty * (size_t)outer_stride);
  const unsigned pst = (unsigned)pt_stride;
  const int tsh = __builtin_ctz(TX);  // TX is a power of two (pick_fft_tiles)
  // forward, first half: unit (l, j2), column j2 + N2 j1 loaded from HBM
  for (int u0 = 0; u0 < N2 * TX; u0 += kBlock) {
    const int u = u0 + tid;
    const int j2 = (u >> tsh);
    const int l = u - j2 * TX;
    const bool live = u < N2 * TX;
    float2 x[N1];
    const unsigned o = (unsigned)j2 * pst + (unsigned)l;
#pragma unroll
    for (int j1 = 0; j1 < N1; j1++)
      x[j1] = (live && l < nl) ? tile[o + (unsigned)(N2 * j1) * pst] : make_float2(0.f, 0.f);
    if (u0 == 0) __syncthreads();  // twiddles in LDS (uniform branch)
    if (live) {
      DftN<N1, -1>::run(x);
#pragma unroll
      for (int k1 = 0; k1 < N1; k1++) {
        const float2 y = k1 == 0 ? x[0] : cmul(x[k1], tw[mul24(j2 * k1, ts)]);
        b[(k1 * N2 + j2) * TX + l] = y;
      }
    }
  }
  __syncthreads();
  double acc[7] = {0, 0, 0, 0, 0, 0, 0};
  zsolve_middle<N1, N2, TRIC>(b, tw, ts, TX, kx0, nl, hxd, sa, acc);
  __syncthreads();
  // inverse second half: unit (l, j2), stored straight to HBM
  for (int u = tid; u < N2 * TX; u += kBlock) {
    const int j2 = (u >> tsh);
    const int l = u - j2 * TX;
    float2 z[N1];
#pragma unroll
    for (int k1 = 0; k1 < N1; k1++) z[k1] = b[(k1 * N2 + j2) * TX + l];
    DftN<N1, +1>::run(z);  // z[j1]: point j = j2 + N2 j1
    if (l < nl) {
      const unsigned o = (unsigned)j2 * pst + (unsigned)l;
#pragma unroll
      for (int j1 = 0; j1 < N1; j1++) store_through(&tile[o + (unsigned)(N2 * j1) * pst], z[j1]);
    }
  }
  if (sa.calc_ev) ev_partial(sa, acc, sh_red, blk);
}

// N2 of the split-precision z lengths 16 N2 (radix_plan_split)
#define PME_ZSOLVE_SPLIT_LENGTHS(X) X(2) X(3) X(4) X(5) X(6) X(8) X(9) X(10) X(12) X(16)

// The same tile for a split-precision z axis of n = 16 N2: the 16-point DFTs as
// hi-lo products on the matrix cores, 32 units per wave, lanes along l.  They come
// first in both directions: the hi-lo error goes with the largest value of a
// 16-point column, and behind the other factor a column of the inverse mixes large
// and small frequencies (250,002 atoms, 144^3, BF16x3: forces 3.83e-5 from FP64 that
// way with one LDS exchange less and 20.9 us, 3.79e-5 this way in 23.1 us; FP32 transforms
// 3.48e-5).  So the inverse splits k = k2 + N2 k1, j = j1 + 16 j2, and
// the buffer holds the spectrum in natural order between the two:
//   1  HBM -> DFT_16 over j1 of j2 + N2 j1, twiddle -> slot k1 + 16 j2
//   2  slots k1 + 16 j2 -> DFT_N2, influence function -> slot k3 = k1 + 16 k2, in place
//   3  slots k2 + N2 k1 -> DFT_16 over k1, twiddle -> slot k2 + N2 j1, in place
//   4  slots k2 + N2 j1 -> DFT_N2 -> HBM, points j1 + 16 j2
template <int N2, int PREC>
__device__ __forceinline__ void zsolve_four_step_split(float2* __restrict__ cg, int hx, int TX, long long pt_stride,
                                                       long long outer_stride, const AxisArgs& ax,
                                                       const SolveArgs& sa, int tx, int ty, int blk, float2* sm,
                                                       int hxd) {
  __shared__ double sh_red[7 * (kBlock / 64)];
  const int tid = threadIdx.x;
  float2* tw = sm;
  float2* b = sm + ax.ntw;
  for (int i = tid; i < ax.ntw; i += kBlock) tw[i] = ax.tw[i];
  const int ts = ax.rp.tstride;
  const int kx0 = tx * TX;
  const int nl = min(TX, hx - kx0);
  float2* __restrict__ tile = cg + ((size_t)kx0 + (size_t)ty * (size_t)outer_stride);
  const unsigned pst = (unsigned)pt_stride;
  const int tsh = __builtin_ctz(TX);
  struct Unit {
    unsigned o;  // point q of the line
    int l, q;
    bool live;
  };
  auto unit = [&](int u) {
    const int q = u >> tsh, l = u - q * TX;
    return Unit{(unsigned)q * pst + (unsigned)l, l, q, l < nl};
  };
  __syncthreads();  // twiddles in LDS
  mfma_dft16_cols<-1, PREC>(
      N2 * TX, unit,
      [&](const Unit& x, int m) { return x.live ? tile[x.o + (unsigned)(N2 * m) * pst] : make_float2(0.f, 0.f); },
      [&](const Unit& x, int k1, float2 y) {
        b[(k1 + 16 * x.q) * TX + x.l] = k1 == 0 ? y : cmul(y, tw[mul24(x.q * k1, ts)]);
      },
      tid, kBlock);
  __syncthreads();
  double acc[7] = {0, 0, 0, 0, 0, 0, 0};
  for (int u = tid; u < 16 * TX; u += kBlock) {
    const int k1 = u >> tsh, l = u - k1 * TX;
    float2 X[N2];
#pragma unroll
    for (int j2 = 0; j2 < N2; j2++) X[j2] = b[(k1 + 16 * j2) * TX + l];
    DftN<N2, -1>::run(X);
    if (l < nl) solve_line_points<16, N2, false>(sa, X, k1, kx0 + l, hxd, acc);
#pragma unroll
    for (int k2 = 0; k2 < N2; k2++) b[(k1 + 16 * k2) * TX + l] = X[k2];
  }
  __syncthreads();
  mfma_dft16_cols<+1, PREC>(
      N2 * TX, unit, [&](const Unit& x, int m) { return b[(x.q + N2 * m) * TX + x.l]; },
      [&](const Unit& x, int j1, float2 y) {
        const float2 t = tw[mul24(x.q * j1, ts)];
        b[(x.q + N2 * j1) * TX + x.l] = j1 == 0 ? y : cmul(y, make_float2(t.x, -t.y));
      },
      tid, kBlock);
  __syncthreads();
  for (int u = tid; u < 16 * TX; u += kBlock) {
    const int j1 = u >> tsh, l = u - j1 * TX;
    float2 X[N2];
#pragma unroll
    for (int k2 = 0; k2 < N2; k2++) X[k2] = b[(k2 + N2 * j1) * TX + l];
    DftN<N2, +1>::run(X);
    if (l < nl) {
      const unsigned o = (unsigned)j1 * pst + (unsigned)l;
#pragma unroll
      for (int j2 = 0; j2 < N2; j2++) store_through(&tile[o + (unsigned)(16 * j2) * pst], X[j2]);
    }
  }
  if (sa.calc_ev) ev_partial(sa, acc, sh_red, blk);
}

}  // namespace pme
