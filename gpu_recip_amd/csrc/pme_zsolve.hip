// pme_zsolve.hip -- the fused z pass (z forward, influence function with energy
// and virial, z inverse in one read and one write of the spectrum) for every
// four-step factor pair, single-system and batched.
#include "pme_zpass.hpp"

namespace pme {

int four_step_code(int n) {
#define PME_F4_CODE(c, a, b) \
  if (n == (a) * (b)) return c;
  PME_F4_PAIRS(PME_F4_CODE)
  PME_F4_Z_PAIRS(PME_F4_CODE)
#undef PME_F4_CODE
  return -1;
}

int four_step_code_for_plan(const RadixPlan& rp) {
  const int code = four_step_code(rp.n);
  int a = 0, b = 0;
  return (rp.f4a > 0 && code >= 0 && four_step_pair(code, &a, &b) && a == rp.f4a && b == rp.f4b) ? code : -1;
}

bool four_step_pair(int code, int* n1, int* n2) {
#define PME_F4_PAIR(c, a, b) \
  if (code == (c)) {         \
    *n1 = (a);               \
    *n2 = (b);               \
    return true;             \
  }
  PME_F4_PAIRS(PME_F4_PAIR)
  PME_F4_Z_PAIRS(PME_F4_PAIR)
#undef PME_F4_PAIR
  return false;
}

int four_step_class(int code) {
#define PME_F4_CLS(c, a, b) \
  if (code == (c)) return f4_class_of(a, b);
  PME_F4_PAIRS(PME_F4_CLS)
  PME_F4_Z_PAIRS(PME_F4_CLS)
#undef PME_F4_CLS
  return -1;
}

// The fused z pass of one grid as a register four-step with n = N1 N2 (one
// kernel per pair, so each gets the registers of its own pair only): column
// tiles of TX lines of the flattened (ky, kx) of a z plane.
// TRIC: triclinic box (90 x 80 x 96 with energy and virial: 104 us per solve with the
// stand-alone scalar sum between a z forward and a z inverse pass, 89 with this).
template <int N1, int N2, bool TRIC>
__global__ __launch_bounds__(kBlock) void k_zsolve(float2* __restrict__ cg, int nlines, int TX, long long pt_stride,
                                                   AxisArgs ax, SolveArgs sa, EvReduce red, int hxd) {
  extern __shared__ __align__(16) float2 sm[];
  if ((red.nsolve > 0 || red.nself > 0) && blockIdx.x == 0) ev_reduce_block<kBlock>(red);
  zsolve_four_step<N1, N2, TRIC>(cg, nlines, TX, pt_stride, 0, ax, sa, blockIdx.x, 0, blockIdx.x, sm, hxd);
}

hipError_t launch_zsolve(float2* cg, int nlines, int TX, long long pt_stride, const AxisArgs& ax, const SolveArgs& sa,
                         const EvReduce& red, int hxd, size_t lds, hipStream_t s) {
  const dim3 g((nlines + TX - 1) / TX), b(kBlock);
  switch (ax.f4) {
#define PME_ZS_CASE(c, n1, n2)                                                                                   \
  case c:                                                                                                        \
    if (sa.tric)                                                                                                 \
      hipLaunchKernelGGL((k_zsolve<n1, n2, true>), g, b, lds, s, cg, nlines, TX, pt_stride, ax, sa, red, hxd);   \
    else                                                                                                         \
      hipLaunchKernelGGL((k_zsolve<n1, n2, false>), g, b, lds, s, cg, nlines, TX, pt_stride, ax, sa, red, hxd);  \
    break;
    PME_F4_PAIRS(PME_ZS_CASE)
    PME_F4_Z_PAIRS(PME_ZS_CASE)
#undef PME_ZS_CASE
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// The split-precision z pass of one grid, one kernel per length and precision
// (one kernel for all of them takes 2.6 us more at 144^3, three waves per SIMD).
template <int N2, int PREC>
__global__ __launch_bounds__(kBlock, 4) void k_zsolve_split(float2* __restrict__ cg, int nlines, int TX,
                                                            long long pt_stride, AxisArgs ax, SolveArgs sa,
                                                            EvReduce red, int hxd) {
  extern __shared__ __align__(16) float2 sm[];
  if ((red.nsolve > 0 || red.nself > 0) && blockIdx.x == 0) ev_reduce_block<kBlock>(red);
  zsolve_four_step_split<N2, PREC>(cg, nlines, TX, pt_stride, 0, ax, sa, blockIdx.x, 0, blockIdx.x, sm, hxd);
}

hipError_t launch_zsolve_split(float2* cg, int nlines, int TX, long long pt_stride, const AxisArgs& ax,
                               const SolveArgs& sa, const EvReduce& red, int hxd, size_t lds, hipStream_t s) {
  const dim3 g((nlines + TX - 1) / TX), b(kBlock);
  if (ax.rp.f4a != 16 || ax.prec == PREC_FP32) return hipErrorInvalidValue;
  switch (ax.rp.f4b) {
#define PME_ZSS_CASE(n2)                                                                                           \
  case n2:                                                                                                         \
    if (ax.prec == PREC_BF16X3)                                                                                    \
      hipLaunchKernelGGL((k_zsolve_split<n2, PREC_BF16X3>), g, b, lds, s, cg, nlines, TX, pt_stride, ax, sa, red, hxd); \
    else                                                                                                           \
      hipLaunchKernelGGL((k_zsolve_split<n2, PREC_FP16X3>), g, b, lds, s, cg, nlines, TX, pt_stride, ax, sa, red, hxd); \
    break;
    PME_ZSOLVE_SPLIT_LENGTHS(PME_ZSS_CASE)
#undef PME_ZSS_CASE
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// ---- batched --------------------------------------------------------------------

// the pairs of register class CLS only
template <int CLS>
__device__ __forceinline__ void zsolve_four_step_dispatch(int code, float2* __restrict__ cg, int hx, int TX,
                                                          long long pt_stride, long long outer_stride,
                                                          const AxisArgs& ax, const SolveArgs& sa, int tx, int ty,
                                                          int blk, float2* sm, int hxd) {
  switch (code) {
#define PME_F4_CASE(c, a, b)                                                                          \
  case c:                                                                                             \
    if constexpr (f4_class_of(a, b) == CLS)                                                              \
      zsolve_four_step<a, b>(cg, hx, TX, pt_stride, outer_stride, ax, sa, tx, ty, blk, sm, hxd);      \
    break;
    PME_F4_PAIRS(PME_F4_CASE)
    PME_F4_Z_PAIRS(PME_F4_CASE)
#undef PME_F4_CASE
    default: break;
  }
}

// The fused z pass of systems whose z length has a four-step pair of class
// CLS (their items only): tiles of the flattened (ky, kx) of a z plane.
template <int CLS>
__global__ __launch_bounds__(kBlock, CLS < 2 ? 4 : 2) void k_batch_zsolve(const SysDesc* __restrict__ sys,
                                                         const WorkItem* __restrict__ items, int nitems) {
  extern __shared__ __align__(16) float2 sm[];
  for (int it = blockIdx.x; it < nitems; it += gridDim.x) {
    const WorkItem w = uniform_item(items[it]);
    const SysDesc& d = sys[w.sys];
    const int hx = d.bin.nx / 2 + 1;
    zsolve_four_step_dispatch<CLS>(d.ax[2].f4, d.cgrid, hx * d.bin.ny, d.TXz, spec_pitch(hx, d.bin.ny), 0, d.ax[2],
                                   d.sa, w.idx, 0, w.idx, sm, hx);
    __syncthreads();
  }
}

hipError_t launch_batch_zsolve(int cls, const SysDesc* sys, const WorkItem* items, int nitems, int grid, size_t lds,
                               hipStream_t s) {
  if (nitems <= 0) return hipSuccess;
  if (cls == 0)
    hipLaunchKernelGGL(k_batch_zsolve<0>, dim3(grid), dim3(kBlock), lds, s, sys, items, nitems);
  else if (cls == 1)
    hipLaunchKernelGGL(k_batch_zsolve<1>, dim3(grid), dim3(kBlock), lds, s, sys, items, nitems);
  else if (cls == 2)
    hipLaunchKernelGGL(k_batch_zsolve<2>, dim3(grid), dim3(kBlock), lds, s, sys, items, nitems);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

// one spectrum times a factor (planes of pitch pz, n used points each)
__global__ __launch_bounds__(kBlock) void k_scale_spectrum(float2* __restrict__ cg, int n, long long pz, float f) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) {
    float2* p = cg + (size_t)blockIdx.y * (size_t)pz + i;
    *p = cscale(*p, f);
  }
}
hipError_t launch_scale_spectrum(float2* cg, int hx, int ny, int nz, float f, hipStream_t s) {
  const int n = hx * ny;
  hipLaunchKernelGGL(k_scale_spectrum, dim3((n + kBlock - 1) / kBlock, nz), dim3(kBlock), 0, s, cg, n,
                     spec_pitch(hx, ny), f);
  return hipGetLastError();
}

}  // namespace pme
