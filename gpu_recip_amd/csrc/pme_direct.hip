// pme_direct.hip -- the direct-space (real-space) half of the Ewald sum for
// CDNA4: the non-bonded pair kernel over the reference's tile neighbour list
// and the 1-4 interaction / exclusion kernel, with the semantics of
// CudaPMEDirectForce<long long, float> (CudaDirectForce_util.h:184-251,
// CudaDirectForceKernels.cu:352-400, 506-716).
//
// Non-bonded pairs.  The waves take the list's j tiles two at a time from a few
// queues as they finish, so the waves' loads even out whatever the spread of the
// tiles' pair counts; a small kernel first maps every j tile to its entry.  Each
// half of a wave takes one tile per pass, one j atom per lane, holding the i tile
// of the tile's entry (32 atoms, moved by the entry's periodic shift on the j
// side) in LDS and flushing the i-force sums whenever the entry changes (with
// tiles from a queue, on most passes).  A pass has two phases.  The check phase
// tests the 32 x 64 pairs against the cutoff, each lane reading the i atoms at LDS
// addresses common to its half (broadcast reads) and building a 32-bit mask of
// its interacting i atoms; rotated into the bit order of the tile's exclusion
// words, the mask loses the excluded pairs.  The dense phase packs the wave's
// interacting pairs into an LDS queue (bit round by bit round, each round a ballot,
// so that 64 consecutive pairs belong to different j atoms) and evaluates them 64 at
// a time, so the Ewald term runs only for pairs inside the cutoff (about one check
// in eight for a 32-atom tile list).  Pair forces are rounded once to 2^40 fixed
// point and summed with integer LDS atomics per i and per j atom; the sums go to
// the caller's force array as integer atomics, the j sums after every pass and the
// i sums when the entry changes, and the shift forces of the virial are summed the
// same way: none of these depends on the order of the pairs.  Pair energies are
// summed as 2^32 fixed point.  Which workgroup takes which tiles varies from run to
// run, so the workgroups' partials stay integers until one reduction has added them
// all and converts the sum once.
#include "pme_internal.hpp"

namespace pme {

// calc_box_shift<float>, gpu_utils.h:312-320: ish = (ix+1) + 3(iy+1) + 9(iz+1)
__device__ __forceinline__ void box_shift(int ish, const DirectParams& d, float& sx, float& sy, float& sz) {
  const int iz = ish / 9, r = ish - 9 * iz, iy = r / 3, ix = r - 3 * iy;
  sx = (float)(ix - 1) * d.boxx;
  sy = (float)(iy - 1) * d.boxy;
  sz = (float)(iz - 1) * d.boxz;
}

// erfc(x) for x >= 0 from e^{-x^2}: erfc(x) e^{x^2} = t P(t) with
// t = 1 / (1 + p x), the form of Hastings' approximation (Abramowitz &
// Stegun 7.1.26) with ten terms whose coefficients were fitted here by
// minimax least squares on the relative error of erfc(x) e^{x^2} over
// [0, 12].  Evaluated in FP32 with the hardware reciprocal its relative error
// is below 4e-7 on [0, 6] (about three ulp, checked against an FP64 erfc).
// The pair term needs e^{-x^2} for the force anyway, so erfc costs a
// reciprocal and ten FMAs.
constexpr float kErfcP = 0.57f;
constexpr float kErfcC[10] = {0.3215866983f,  0.3216636181f, 0.2678903937f, 0.1791002899f,  -0.0476588681f,
                              0.2127946466f,  -0.7263579965f, 0.7648586631f, -0.3605679274f, 0.0666905344f};
__device__ __forceinline__ float erfc_from_exp(float x, float exp_neg_x2) {
  const float t = __builtin_amdgcn_rcpf(fmaf(kErfcP, x, 1.0f));
  float acc = kErfcC[9];
#pragma unroll
  for (int k = 8; k >= 0; k--) acc = fmaf(acc, t, kErfcC[k]);
  return acc * t * exp_neg_x2;
}

// e^{-x} for x >= 0: 2^(-x log2 e) by the hardware exponential (1 ulp) with
// the product's rounding error and the low part of log2 e carried into a
// correction factor, so that the result is good to about 1 ulp for every x (the
// plain product loses x/2 ulp); results below the normal range are 0.
__device__ __forceinline__ float exp_neg(float x) {
  const float l2e = 1.44269504f, l2e_lo = 1.92596299e-8f, ln2 = 0.693147181f;
  const float t = x * l2e;
  const float lo = fmaf(x, l2e_lo, fmaf(x, l2e, -t));
  const float y = __builtin_amdgcn_exp2f(-t);
  return fmaf(y, -lo * ln2, y);
}

// The EWALD pair term (CudaDirectForceKernels.cu:352-390) for charges already
// multiplied by ccelec: pot = qq (erfc(kappa r) + fac_m1) / r with fac_m1 = 0
// for non-bonded pairs, e14fac - 1 for 1-4 interactions and -1 for 1-4
// exclusions.  Returns fij = (r dU/dr) / r^2, so that fij * (xi - xj) is the
// gradient on i.
__device__ __forceinline__ float ewald_fij(float r2, float rinv, float qq, float fac_m1, const DirectParams& d,
                                           float& pot) {
  const float r = r2 * rinv;
  const float exp_val = exp_neg(d.kappa2 * r2);
  const float erfc_val = erfc_from_exp(d.kappa * r, exp_val);
  const float qq_efac_rinv = qq * (erfc_val + fac_m1) * rinv;
  pot = qq_efac_rinv;
  const float two_sqrtpi = 1.12837916709551f;  // 2/sqrt(pi)
  const float fij_elec = -qq * two_sqrtpi * d.kappa * exp_val - qq_efac_rinv;
  return fij_elec * rinv * rinv;
}

// f (+=) as 2^40 fixed point, write_force<long long> (gpu_utils.h:292-302)
__device__ __forceinline__ void add_fixed(unsigned long long* force, int i, int stride, float fx, float fy, float fz) {
  atomicAdd(&force[i], (unsigned long long)(long long)rintf(kForceScale * fx));
  atomicAdd(&force[(size_t)i + stride], (unsigned long long)(long long)rintf(kForceScale * fy));
  atomicAdd(&force[(size_t)i + 2 * (size_t)stride], (unsigned long long)(long long)rintf(kForceScale * fz));
}

// A pair-force component as 2^40 fixed point, rounded once to the nearest
// integer.  Below 2^11 in magnitude (every pair outside close contact) one
// FMA does it (to_fixed_product: f * 2^40 is exact in FP64 and below 2^51);
// larger f * 2^40 are integers already and convert exactly, held inside the
// format's range of +-2^23.
__device__ __forceinline__ unsigned long long pair_fixed(float f) {
  if (fabsf(f) < 2048.0f) return to_fixed_product((double)f, 1099511627776.0);
  const float c = fminf(fmaxf(f, -8388607.0f), 8388607.0f);
  return (unsigned long long)(long long)((double)c * 1099511627776.0);
}

// The force of a pair and its negative: one range test for the three components,
// and the negative of the integer where the rounding is to nearest even (which is
// symmetric).
__device__ __forceinline__ void pair_fixed3(const float* f, unsigned long long* gi, unsigned long long* gj) {
  const bool small = fmaxf(fmaxf(fabsf(f[0]), fabsf(f[1])), fabsf(f[2])) < 2048.0f;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    gi[c] = to_fixed_product((double)f[c], 1099511627776.0);
    gj[c] = 0ull - gi[c];
  }
  if (!small) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      gi[c] = pair_fixed(f[c]);
      gj[c] = pair_fixed(-f[c]);
    }
  }
}

// A pair energy as 2^32 fixed point (integer sums do not depend on which wave
// takes which pairs); |e| < 2^19 by one FMA, larger ones held inside +-2^30.
__device__ __forceinline__ long long energy_fixed(float e) {
  if (fabsf(e) < 524288.0f) return (long long)to_fixed_product((double)e, 4294967296.0);
  const float c = fminf(fmaxf(e, -1073741824.0f), 1073741824.0f);
  return (long long)((double)c * 4294967296.0);
}

// Orders the LDS accesses of the lanes of one wave (all of them issue from
// the same instruction stream, so a compiler barrier and the LDS counter wait
// are enough; no workgroup barrier).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The workgroup's partials: elec, excl, then sforce[27][3] (the shift forces
// of the virial, CudaEnergyVirial.h:14).  Each thread brings its energies and
// one shift-force contribution (ish < 0: none); the energies are summed with
// block_sum in fixed order, the shift forces per shift as 2^40 fixed point
// with integer LDS atomics (exact, so the order does not matter).
template <int NT>
__device__ __forceinline__ void write_direct_partial(double elec, double excl, int ish, float sfx, float sfy,
                                                     float sfz, bool energy, bool virial, double* out, size_t st) {
  __shared__ double s_red[2 * (NT / 64)];
  __shared__ unsigned long long s_sf[81];
  const int tid = threadIdx.x;
  if (virial) {
    for (int k = tid; k < 81; k += NT) s_sf[k] = 0ull;
    __syncthreads();
    if (ish >= 0) {
      atomicAdd(&s_sf[3 * ish + 0], pair_fixed(sfx));
      atomicAdd(&s_sf[3 * ish + 1], pair_fixed(sfy));
      atomicAdd(&s_sf[3 * ish + 2], pair_fixed(sfz));
    }
  }
  if (energy) {
    double v[2] = {elec, excl};
    block_sum<2, NT>(v, s_red);
    if (tid == 0) {
      out[0] = v[0];
      out[st] = v[1];
    }
  }
  if (virial) {
    __syncthreads();
    for (int k = tid; k < 81; k += NT) out[(2 + k) * st] = (double)(long long)s_sf[k] * (1.0 / 1099511627776.0);
  }
}

// tile_entry[t] = -1 for every tile (the map kernel then fills in the tiles
// of the entries), and the chunk queues of the pair kernel to zero.
__global__ __launch_bounds__(256) void k_direct_tile_clear(int n_tile, int* __restrict__ tile_entry,
                                                           int* __restrict__ queue) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t < n_tile) tile_entry[t] = -1;
  if (t < kDirQueues) queue[t * kDirQueuePad] = 0;
}

// Every j tile's entry: tile_entry[t] = e for tileStart <= t <= tileEnd of
// entry e, one wave per entry; tiles of no entry stay -1.
__global__ __launch_bounds__(256) void k_direct_tile_map(int n_ientry, const pme_ientry* __restrict__ ientry,
                                                         int n_tile, int* __restrict__ tile_entry) {
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (e >= n_ientry) return;
  const pme_ientry en = ientry[e];
  const int hi = min(en.tileEnd, n_tile - 1);
  for (int t = max(en.tileStart, 0) + lane; t <= hi; t += 64) tile_entry[t] = e;
}

// A coordinate, or `far` in place of a NaN or an infinity: the check phase reads
// the sign of r^2 - roff^2, which a NaN has too; i and j atoms get far values of
// opposite sign, so no such pair is inside the cutoff.
__device__ __forceinline__ float far_or(float x, float far) { return fabsf(x) < 1e18f ? x : far; }

// LDS of one wave of the pair kernel
struct DirWave {
  float4 xi[2][33];                 // i tile of each half's entry, q * ccelec (rows padded: other banks)
  float4 xj[64];                    // j atoms of the pass moved by minus their shift, q
  unsigned long long fi[2][3][32];  // i force sums of each half's entry, 2^40 fixed point
  unsigned long long fj[3][64];     // j force sums of the pass
  unsigned short pairs[32 * 64];    // interacting pairs of the pass: i | (j lane << 5)
};

// Adds the i-force sums of a half's entry to the force array and, for a
// shifted image, to the shift forces; clears them.  Lanes of the half only.
template <bool VIRIAL>
__device__ __forceinline__ void flush_entry(DirWave& W, int h, int jl, int iatom, int ish, int stride,
                                            unsigned long long* __restrict__ force, unsigned long long* s_sf) {
  unsigned long long g[3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    g[c] = W.fi[h][c][jl];
    W.fi[h][c][jl] = 0ull;
  }
  if (g[0] | g[1] | g[2]) {
    atomicAdd(&force[iatom + jl], g[0]);
    atomicAdd(&force[(size_t)(iatom + jl) + stride], g[1]);
    atomicAdd(&force[(size_t)(iatom + jl) + 2 * (size_t)stride], g[2]);
    // the entry's shift force (CudaDirectForce_util.h:321-347): the sum of
    // its i forces, except for the central image
    if (VIRIAL && ish != 13) {
#pragma unroll
      for (int c = 0; c < 3; c++) atomicAdd(&s_sf[3 * ish + c], g[c]);
    }
  }
}

// The list's j tiles in pairs, one tile per half of a wave and pass.  A wave
// starts with its own pair of tiles and takes the following ones from a queue:
// atomics of all XCDs on one address complete about one in 20 ns, so there are
// kDirQueues of them, each in a cache line of its own, queue q holding the pairs
// q, q + kDirQueues, ... (every queue sees tiles from the whole list, whose pair
// density varies tenfold).  The queue runs two pairs ahead: while one is
// processed, the tile records (entry, atom index, exclusions) of the next are
// loaded and the ticket of the one after it is under way.  Chunks of 8 tiles
// dealt to the waves in turn took 91 us for 24,000 atoms (roff 9 A, 33,273 tiles;
// the mean CU was busy for 57 of them) and 268 us for 96,000; the queue with
// chunks of 8, 4 and 2 tiles takes 77, 73, 67 and 199, 183, 180 us.
template <bool ENERGY, bool VIRIAL>
__global__ __launch_bounds__(kDirWaves * 64) void k_direct_force(DirectParams d, int n_ientry, int n_tile,
                                                                 const pme_ientry* __restrict__ ientry,
                                                                 const int* __restrict__ tile_entry,
                                                                 int* __restrict__ queue,
                                                                 const int* __restrict__ tile_indj,
                                                                 const pme_tile_excl* __restrict__ tile_excl,
                                                                 const float4* __restrict__ xyzq, int stride,
                                                                 unsigned long long* __restrict__ force,
                                                                 double* __restrict__ partial) {
  __shared__ DirWave s_w[kDirWaves];
  __shared__ unsigned long long s_sf[81];  // shift forces, 2^40 fixed point
  __shared__ unsigned long long s_pot;     // energy, 2^32 fixed point
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, h = lane >> 5, jl = lane & 31;
  DirWave& W = s_w[wv];
  if (threadIdx.x < 81) s_sf[threadIdx.x] = 0ull;
  if (threadIdx.x == 0) s_pot = 0ull;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    W.fi[h][c][jl] = 0ull;
    W.fj[c][lane] = 0ull;
  }
  __syncthreads();
  const int nchunk = (n_tile + 1) >> 1;  // pairs of tiles
  // waves and queues (at least one wave per queue)
  const int wtotal = (int)gridDim.x * kDirWaves;
  const int nq = min(kDirQueues, wtotal);
  const int w0 = (int)blockIdx.x * kDirWaves + wv, q0 = w0 % nq;
  const int first = q0 + nq * ((wtotal - q0 + nq - 1) / nq);  // first chunk of the queue that no wave starts with
  int* const ctr = queue + q0 * kDirQueuePad;
  int chunk = w0;
  int ticket = 0;  // lane 0
  // the half's current entry
  int cur = -1, cur_lo = 0, cur_hi = -1, cur_ish = 13, cur_i0 = 0;
  float sx = 0.f, sy = 0.f, sz = 0.f;
  long long pot = 0;
  // tile record of the half's tile of a pair
  int ne = -1, nindj = 0;
  unsigned nexcl = 0xffffffffu;
  auto load_record = [&](int c) {
    const int t = 2 * c + h;
    const bool in = c < nchunk && t < n_tile;
    ne = in ? tile_entry[t] : -1;
    nindj = in ? tile_indj[t] : 0;
    nexcl = in ? tile_excl[t].excl[jl] : 0xffffffffu;
  };
  auto take = [&]() {
    if (lane == 0) ticket = atomicAdd(ctr, 1);
  };
  take();
  load_record(chunk);
  while (chunk < nchunk) {
    const int t = 2 * chunk + h;
    const int e = ne, indj = nindj;
    const unsigned excl = nexcl;
    // the j atoms of this pass, then the record of the next one
    const float4 pj = e >= 0 ? xyzq[indj + jl] : make_float4(0.f, 0.f, 0.f, 0.f);
    const int next = first + nq * __builtin_amdgcn_readfirstlane(ticket);
    if (next < nchunk) take();
    load_record(next);
    if (e != cur) {
      if (cur >= 0) flush_entry<VIRIAL>(W, h, jl, cur_i0, cur_ish, stride, force, s_sf);
      cur = -1;
      if (e >= 0 && e < n_ientry) {
        const pme_ientry en = ientry[e];
        if (t >= en.tileStart && t <= en.tileEnd) {
          cur = e;
          cur_lo = en.tileStart;
          cur_hi = en.tileEnd;
          cur_ish = en.ish;
          cur_i0 = en.iatomStart;
          box_shift(cur_ish, d, sx, sy, sz);
          const float4 p = xyzq[cur_i0 + jl];
          W.xi[h][jl] = make_float4(far_or(p.x, 1e18f), far_or(p.y, 1e18f), far_or(p.z, 1e18f), p.w * (float)kCcelec);
        }
      }
    }
    wave_lds_sync();
    const bool ok = cur >= 0 && t >= cur_lo && t <= cur_hi && t < n_tile;
    // xi - (xj - shift) is the separation of i's image from j
    const float xjx = far_or(pj.x - sx, -1e18f), xjy = far_or(pj.y - sy, -1e18f), xjz = far_or(pj.z - sz, -1e18f);
    W.xj[lane] = make_float4(xjx, xjy, xjz, pj.w);
    // check phase: bit i of m = pair (i, j) inside the cutoff
    unsigned m = 0u;
#pragma unroll
    for (int g = 3; g >= 0; g--) {
      float4 pg[8];  // eight i atoms read together, then tested
#pragma unroll
      for (int u = 0; u < 8; u++) pg[u] = W.xi[h][8 * g + u];
#pragma unroll
      for (int u = 7; u >= 0; u--) {
        // the sign of r^2 - roff^2, shifted into m
        const float dx = pg[u].x - xjx, dy = pg[u].y - xjy, dz = pg[u].z - xjz;
        const float s = fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, -d.roff2)));
        m = __builtin_amdgcn_alignbit(m, __float_as_uint(s), 31);
      }
    }
    // rotated right by l, bit t of m is i = (l + t) mod 32, as in the exclusion word excl[l]
    m = __builtin_amdgcn_alignbit(m, m, jl) & ~excl;
    if (!ok) m = 0u;
    // dense phase: the wave's pairs packed round by round, each lane's next
    // pair per round, so neighbours in the queue have different j atoms, and,
    // each lane counting from its own place in the i tile, mostly different i
    // atoms too: lanes that add to one LDS address wait for each other (24,000
    // atoms, roff 9 A: 67.6 -> 60.3 us; of those 9.5 are the i atomics, 5 the j
    // atomics, 17 the pair terms, 12 the check and packing)
    int total = 0;
    for (;;) {
      const unsigned long long on = __ballot(m != 0u);
      if (on == 0ull) break;
      if (m) {
        const int i = (__ffs(m) - 1 + jl) & 31;
        m &= m - 1u;
        const int slot = total + __builtin_amdgcn_mbcnt_hi((unsigned)(on >> 32),
                                                           __builtin_amdgcn_mbcnt_lo((unsigned)on, 0u));
        W.pairs[slot] = (unsigned short)(i | (lane << 5));  // at most 32 x 64 pairs
      }
      total += __popcll(on);
    }
    wave_lds_sync();
    for (int q = lane; q < total; q += 64) {
      const unsigned pr = W.pairs[q];
      const int i = pr & 31, l = pr >> 5, hl = l >> 5;
      const float4 pi = W.xi[hl][i], pjl = W.xj[l];
      const float dx = pi.x - pjl.x, dy = pi.y - pjl.y, dz = pi.z - pjl.z;
      const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
      float pe;
      const float fij = ewald_fij(r2, rsqrtf(r2), pi.w * pjl.w, 0.0f, d, pe);
      if (ENERGY) pot += energy_fixed(pe);
      const float f[3] = {fij * dx, fij * dy, fij * dz};
      unsigned long long gi[3], gj[3];
      pair_fixed3(f, gi, gj);
#pragma unroll
      for (int c = 0; c < 3; c++) {
        atomicAdd(&W.fi[hl][c][i], gi[c]);
        atomicAdd(&W.fj[c][l], gj[c]);
      }
    }
    wave_lds_sync();
    unsigned long long g[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
      g[c] = W.fj[c][lane];
      W.fj[c][lane] = 0ull;
    }
    if (ok && (g[0] | g[1] | g[2])) {
      atomicAdd(&force[indj + jl], g[0]);
      atomicAdd(&force[(size_t)(indj + jl) + stride], g[1]);
      atomicAdd(&force[(size_t)(indj + jl) + 2 * (size_t)stride], g[2]);
    }
    wave_lds_sync();
    chunk = next;
  }
  if (cur >= 0) flush_entry<VIRIAL>(W, h, jl, cur_i0, cur_ish, stride, force, s_sf);
  if (ENERGY || VIRIAL) {
    if (ENERGY && pot != 0) atomicAdd(&s_pot, (unsigned long long)pot);
    __syncthreads();
    // integers in the partials' places (k_direct_reduce<true>)
    long long* out = reinterpret_cast<long long*>(partial) + blockIdx.x;
    const size_t st = gridDim.x;
    const int tid = threadIdx.x;
    if (ENERGY && tid == 0) {
      out[0] = (long long)s_pot;
      out[st] = 0;
    }
    if (VIRIAL && tid < 81) out[(2 + tid) * st] = (long long)s_sf[tid];
  }
}

// 1-4 interactions [0, nin14) and exclusions [nin14, nin14 + nex14), one
// entry per thread (calc_14_force_kernel, CudaDirectForceKernels.cu:664-760).
template <bool ENERGY, bool VIRIAL>
__global__ __launch_bounds__(kDir14Block) void k_direct_14(DirectParams d, int nin14, int nex14,
                                                           const pme_xx14* __restrict__ in14,
                                                           const pme_xx14* __restrict__ ex14,
                                                           const float4* __restrict__ xyzq, int stride,
                                                           unsigned long long* __restrict__ force,
                                                           double* __restrict__ partial) {
  const int k = blockIdx.x * kDir14Block + threadIdx.x;
  double elec = 0.0, excl = 0.0;
  float sfx = 0.f, sfy = 0.f, sfz = 0.f;
  int ish_out = -1;
  if (k < nin14 + nex14) {
    const bool is_in = k < nin14;
    const pme_xx14 p = is_in ? in14[k] : ex14[k - nin14];
    float sx, sy, sz;
    box_shift(p.ishift, d, sx, sy, sz);
    const float4 xi = xyzq[p.i], xj = xyzq[p.j];
    const float dx = xi.x - xj.x + sx, dy = xi.y - xj.y + sy, dz = xi.z - xj.z + sz;
    const float r2 = dx * dx + dy * dy + dz * dz;
    const float qq = (float)kCcelec * xi.w * xj.w;
    const float r = sqrtf(r2);
    float pe;
    const float fij = ewald_fij(r2, 1.0f / r, qq, is_in ? d.e14fac - 1.0f : -1.0f, d, pe);
    if (is_in) elec = (double)pe;
    else excl = (double)pe;
    const float fx = fij * dx, fy = fij * dy, fz = fij * dz;
    add_fixed(force, p.i, stride, fx, fy, fz);
    add_fixed(force, p.j, stride, -fx, -fy, -fz);
    if (p.ishift != 13) {
      ish_out = p.ishift;
      sfx = fx;
      sfy = fy;
      sfz = fz;
    }
  }
  if (ENERGY || VIRIAL)
    write_direct_partial<kDir14Block>(elec, excl, VIRIAL ? ish_out : -1, sfx, sfy, sfz, ENERGY, VIRIAL,
                                      partial + blockIdx.x, gridDim.x);
}

// Sum of the 64-bit integers v[0], v[1], ... v[n-1] times scale, rounded once: the
// high and the low halves are summed apart, so no total overflows (256 threads; the
// result in thread 0).
__device__ __forceinline__ double block_sum_fixed(const long long* __restrict__ v, int n, double scale) {
  __shared__ unsigned long long s_half[2];
  if (threadIdx.x < 2) s_half[threadIdx.x] = 0ull;
  __syncthreads();
  long long hi = 0, lo = 0;
  for (int b = threadIdx.x; b < n; b += 256) {
    hi += v[b] >> 32;
    lo += v[b] & 0xffffffffll;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    hi += __shfl_xor(hi, off, 64);
    lo += __shfl_xor(lo, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&s_half[0], (unsigned long long)hi);
    atomicAdd(&s_half[1], (unsigned long long)lo);
  }
  __syncthreads();
  const long long h = (long long)s_half[0] + (long long)(s_half[1] >> 32);
  return __fma_rn((double)h, 4294967296.0 * scale, (double)(unsigned)s_half[1] * scale);
}

// Sum the partials of nblk workgroups (slot c of workgroup b at c nblk + b) and add
// them into the energy/virial buffer: the elec and excl slots and
// sforce_dp[27][3].  One workgroup per slot.  FIXED: the pair kernel's integers
// (energies 2^32, shift forces 2^40 fixed point), whose sum does not depend on the
// order; else FP64 values, thread k summing workgroups k, k + 256, ... and
// block_sum the threads in fixed order.  The same result on every run either way.
template <bool FIXED>
__global__ __launch_bounds__(256) void k_direct_reduce(const double* __restrict__ partial, int nblk, int energy,
                                                       int virial, double* e_elec, double* e_excl,
                                                       double* sforce_dp) {
  __shared__ double s_red[4];
  const int c = blockIdx.x;
  if ((c < 2 && !energy) || (c >= 2 && !virial)) return;
  double acc = 0.0;
  if (FIXED) {
    acc = block_sum_fixed(reinterpret_cast<const long long*>(partial) + (size_t)c * nblk, nblk,
                          c < 2 ? 1.0 / 4294967296.0 : 1.0 / 1099511627776.0);
  } else {
    for (int b = threadIdx.x; b < nblk; b += 256) acc += partial[(size_t)c * nblk + b];
    block_sum<1, 256>(&acc, s_red);
  }
  if (threadIdx.x == 0) {
    if (c == 0) e_elec[0] += acc;
    else if (c == 1) e_excl[0] += acc;
    else sforce_dp[c - 2] += acc;
  }
}

hipError_t launch_direct_force(const DirectParams& d, int n_ientry, int n_tile, int nwave,
                               const pme_ientry* ientry, int* queue, int* tile_entry, const int* tile_indj,
                               const pme_tile_excl* tile_excl, const float4* xyzq, int stride,
                               unsigned long long* force, bool energy, bool virial, double* partial,
                               hipStream_t s) {
  if (n_ientry <= 0 || n_tile <= 0 || nwave <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_direct_tile_clear, dim3((n_tile + 255) / 256), dim3(256), 0, s, n_tile, tile_entry, queue);
  hipLaunchKernelGGL(k_direct_tile_map, dim3((n_ientry + 3) / 4), dim3(256), 0, s, n_ientry, ientry, n_tile,
                     tile_entry);
  const dim3 g(direct_force_blocks(nwave));
  const dim3 b(kDirWaves * 64);
  if (energy && virial)
    hipLaunchKernelGGL((k_direct_force<true, true>), g, b, 0, s, d, n_ientry, n_tile, ientry, tile_entry, queue,
                       tile_indj, tile_excl, xyzq, stride, force, partial);
  else if (energy)
    hipLaunchKernelGGL((k_direct_force<true, false>), g, b, 0, s, d, n_ientry, n_tile, ientry, tile_entry, queue,
                       tile_indj, tile_excl, xyzq, stride, force, partial);
  else if (virial)
    hipLaunchKernelGGL((k_direct_force<false, true>), g, b, 0, s, d, n_ientry, n_tile, ientry, tile_entry, queue,
                       tile_indj, tile_excl, xyzq, stride, force, partial);
  else
    hipLaunchKernelGGL((k_direct_force<false, false>), g, b, 0, s, d, n_ientry, n_tile, ientry, tile_entry, queue,
                       tile_indj, tile_excl, xyzq, stride, force, partial);
  return hipGetLastError();
}

hipError_t launch_direct_14(const DirectParams& d, int nin14, int nex14, const pme_xx14* in14, const pme_xx14* ex14,
                            const float4* xyzq, int stride, unsigned long long* force, bool energy, bool virial,
                            double* partial, hipStream_t s) {
  const int nblk = direct_14_blocks(nin14 + nex14);
  if (nblk == 0) return hipSuccess;
  const dim3 g(nblk), b(kDir14Block);
  if (energy && virial)
    hipLaunchKernelGGL((k_direct_14<true, true>), g, b, 0, s, d, nin14, nex14, in14, ex14, xyzq, stride, force, partial);
  else if (energy)
    hipLaunchKernelGGL((k_direct_14<true, false>), g, b, 0, s, d, nin14, nex14, in14, ex14, xyzq, stride, force, partial);
  else if (virial)
    hipLaunchKernelGGL((k_direct_14<false, true>), g, b, 0, s, d, nin14, nex14, in14, ex14, xyzq, stride, force, partial);
  else
    hipLaunchKernelGGL((k_direct_14<false, false>), g, b, 0, s, d, nin14, nex14, in14, ex14, xyzq, stride, force,
                       partial);
  return hipGetLastError();
}

hipError_t launch_direct_reduce(bool fixed, const double* partial, int nblk, bool energy, bool virial, double* e_elec,
                                double* e_excl, double* sforce_dp, hipStream_t s) {
  if (nblk == 0 || !(energy || virial)) return hipSuccess;
  const dim3 g(kDirPartial), b(256);
  const int ce = energy ? 1 : 0, cv = virial ? 1 : 0;
  if (fixed)
    hipLaunchKernelGGL(k_direct_reduce<true>, g, b, 0, s, partial, nblk, ce, cv, e_elec, e_excl, sforce_dp);
  else
    hipLaunchKernelGGL(k_direct_reduce<false>, g, b, 0, s, partial, nblk, ce, cv, e_elec, e_excl, sforce_dp);
  return hipGetLastError();
}

int direct_force_blocks(int nwave) { return (nwave + kDirWaves - 1) / kDirWaves; }

int direct_force_waves(int n_tile, int ncu) {
  // 16 waves per CU (four workgroups of kDirWaves), at most one per pair of tiles
  return std::max(1, std::min(ncu * 16, (n_tile + 1) / 2));
}
int direct_14_blocks(int n) { return (n + kDir14Block - 1) / kDir14Block; }

}  // namespace pme
