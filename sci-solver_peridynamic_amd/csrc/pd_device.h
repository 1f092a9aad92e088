// pd_device.h -- device-side layout and helpers shared by the HIP kernels.
//
// HBM layout (one context, N particles, S = ceil(N/64) slices):
//   * particle vectors: double4 per particle (32 B, w lane 0) so that the
//     gathered x_q of a bond is one aligned 32-byte segment;
//   * bonds: sliced ELL with 64 rows per slice (one wave64 lane per row).
//     Slice s owns slot rows [slice_off[s], slice_off[s+1]); the slot k of
//     row p = 64 s + lane lives at (slice_off[s] + k) * 64 + lane, so the
//     64 lanes of a wave touch 64 consecutive words per slot;
//   * matrix values: the 3x3 blocks are symmetric bit for bit, so six
//     values (a00 a01 a02 a11 a12 a22) are stored.  FP64: in three planes
//     of pairs, so a lane reads 16 bytes per load: value c of slot k of row
//     p at ((slice_off[s] + k) * 3 + c / 2) * 128 + 2 * lane + c % 2.
//     Float copy (val32): 384 floats per slot row, a plane of quads
//     (a00 a01 a02 a11) then a plane of pairs (a12 a22), so a lane reads
//     one 16-byte and one 8-byte word: at (slice_off[s] + k) * 384, the
//     quad at 4 * lane and the pair at 256 + 2 * lane;
//   * diagonal and block-Jacobi inverse blocks: (s * 6 + c) * 64 + lane;
//   * mixed precision keeps float copies in the same positions (val32,
//     diag32, minv32) and float4 vectors (16 B) for the inner solve.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define PD_WAVE 64
#define PD_BLOCK 256  // 4 waves = 4 slices = one reduction tile
#define PD_INVISIBLE 3

struct pd_mat_dev {
  double horizon, radius, c_bond, mass;
};

// Scalars of one CG solve, resident in device memory.
struct pd_cg_state {
  double rz;     // <r, z>
  double yp;     // <A p, p>
  double alpha;
  double beta;
  double rr;     // <r, r>
  double bnorm;  // ||S b||
  double tol;    // rtol * bnorm
  double rnorm;  // sqrt(rr)
  double rtol;
  double upd_rz;  // rz and iter as that update found them
  int32_t iter;
  int32_t done;
  int32_t converged;
  int32_t max_iter;
  int32_t upd_it;  // the iteration whose update ran last (-1: none yet)
  int32_t upd_iter;
  uint32_t pad[2];
};

// Scalars of one mixed-precision solve (iterative refinement around a float
// PCG).  phase: 0 residual due, 1 inner iterations, 2 inner finished
// (correction pending, then residual), 3 done.  Grid kernels only read
// phase; the one-workgroup fold kernels change it.
struct pd_mx_state {
  double rz;         // <r32, z32> (FP64 sum of widened floats)
  double rr32;       // <r32, r32>
  double alpha;
  double beta;
  double rnorm;      // ||S(b - A x)||, FP64
  double bnorm;      // ||S b||
  double tol;        // rtol * bnorm
  double inner_tol;  // max(inner_rtol * rnorm, tol / 2)
  double rtol;
  double inner_rtol;
  int32_t iter;        // inner iterations over the whole solve
  int32_t inner_iter;  // of the current refinement
  int32_t refinements;
  int32_t phase;
  int32_t converged;
  int32_t first;
  int32_t max_iter;
  int32_t inner_max;
  int32_t max_refine;
  int32_t residuals;  // FP64 residual evaluations so far
  int32_t pad[2];
};

// Step scalars read from device memory by captured (graph) steps, so one
// graph serves every step.
struct pd_step_consts {
  double dt;
  double dt2;
  double clock;
  double gravity;
};

// Per-step counters written by the assembly kernel.
struct pd_step_counters {
  unsigned long long broken;
  unsigned long long live;
  // bit 0: some position, reference length, bond stiffness, horizon or
  // radius lies outside the ranges of the shared-reciprocal quotients and
  // of sqrt_rcp (set ahead of the assembly); bit 1: a live bond is no longer
  // than (float)1e-10 (set by the assembly).  Nonzero: the matrix-free operator
  // divides one quotient at a time and takes IEEE square roots.
  unsigned int range_bad;
  unsigned int pad;
};

// The CG updates form alpha = rz / <y, p> in every workgroup from the
// specimen's <y, p> tile partials (one read of the partial row per
// workgroup, hidden behind the row loads); a specimen of more tiles than
// this has alpha folded once, by one workgroup, ahead of the update, since
// the per-workgroup reads grow with the square of its tile count.
#define PD_ALPHA_FOLD_TILES 8192
// Largest system, in tiles, whose direction update folds <r, z> and <r, r>
// itself, in every workgroup, instead of after a one-workgroup kernel: 4.8 us
// for both against 8.6 at 110 tiles, 5.4 against 8.2 at 510, but 41.8 against
// 37.2 at 3930, where the workgroups' reads add up to 250 MB.
#define PD_DIR_FOLD_TILES 1024
// Largest systems, in slices, whose matrix-free product takes four and eight
// lanes per row (k_cg_spmv_lanes).
#define PD_LANES_SLICES 1536
#define PD_LANES8_SLICES 512

__device__ __forceinline__ double4 ld4(const double4* p) { return *p; }

// Blocks of the workgroup grid are handed to the 8 XCDs round-robin; this
// maps the hardware order onto contiguous tile ranges per XCD so that the
// tiles sharing an L2 are neighbours in the particle order.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
  const int xcd = b & 7;
  const int idx = b >> 3;
  const int q = nb >> 3;
  const int r = nb & 7;
  return xcd < r ? xcd * (q + 1) + idx : r * (q + 1) + (xcd - r) * q + idx;
}

// v + (v of the lane M away by xor), the level M of a wave's butterfly sum.
// Within a row of 16 lanes through DPP moves, across rows through the lane
// swaps of gfx950 (both operands of the swap hold v, so in every lane their
// sum is the level's).  A level through the LDS crossbar (__shfl_xor) waits
// about 130 cycles, this one about 30.
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
  const int64_t b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((int64_t)hi << 32) | (uint32_t)lo);
}
// v and the v of the lane M away by xor (a, b: in either order, the same in
// both lanes of a pair when M >= 16)
template <int M>
__device__ __forceinline__ void xor_pair(double v, double& a, double& b) {
  a = v;
  if constexpr (M == 1) b = dpp_mov<0xb1>(v);                  // quad_perm 1 0 3 2
  if constexpr (M == 2) b = dpp_mov<0x4e>(v);                  // quad_perm 2 3 0 1
  if constexpr (M == 4) b = dpp_mov<0x1b>(dpp_mov<0x141>(v));  // i ^ 7, then i ^ 3
  if constexpr (M == 8) b = dpp_mov<0x128>(v);                 // row_ror 8
  if constexpr (M >= 16) {
    const int64_t bits = __double_as_longlong(v);
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    const unsigned int l = (unsigned int)bits, h = (unsigned int)(bits >> 32);
    u2 sl, sh;
    if constexpr (M == 16) {
      sl = __builtin_amdgcn_permlane16_swap(l, l, false, false);
      sh = __builtin_amdgcn_permlane16_swap(h, h, false, false);
    } else {
      sl = __builtin_amdgcn_permlane32_swap(l, l, false, false);
      sh = __builtin_amdgcn_permlane32_swap(h, h, false, false);
    }
    a = __longlong_as_double(((int64_t)sh.x << 32) | sl.x);
    b = __longlong_as_double(((int64_t)sh.y << 32) | sl.y);
  }
}
template <int M>
__device__ __forceinline__ double xor_add(double v) {
  double a, b;
  xor_pair<M>(v, a, b);
  return a + b;
}

// Sum of a double over the 64 lanes by the xor butterfly m = 32..1; every
// lane ends with the same value (the order fixed by the oracle's orc_dot).
__device__ __forceinline__ double wave_sum(double v) {
  v = xor_add<32>(v);
  v = xor_add<16>(v);
  v = xor_add<8>(v);
  v = xor_add<4>(v);
  v = xor_add<2>(v);
  return xor_add<1>(v);
}

// Tile reduction of one value per thread of a 256-thread workgroup:
// (w0 + w1) + (w2 + w3) of the four wave sums.  All threads must call it.
__device__ __forceinline__ double tile_sum(double v, double* lds4) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) lds4[w] = v;
  __syncthreads();
  const double r = (lds4[0] + lds4[1]) + (lds4[2] + lds4[3]);
  __syncthreads();
  return r;
}

// Orders a wave's LDS writes before its own lanes' later reads.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// acc + t[0] + t[1] + .. + t[n - 1], left to right; the next eight terms are
// on their way from LDS while eight are added.
__device__ __forceinline__ double chain_add(double acc, const double* t, int n) {
  double h[8];
  int e = 0;
  if (n >= 8) {
#pragma unroll
    for (int u = 0; u < 8; ++u) h[u] = t[u];
    for (; e + 16 <= n; e += 8) {
      double k[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) k[u] = t[e + 8 + u];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += h[u];
#pragma unroll
      for (int u = 0; u < 8; ++u) h[u] = k[u];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) acc += h[u];
    e += 8;
  }
  for (; e < n; ++e) acc += t[e];
  return acc;
}

// tile_sum of N quantities, one exchange; lds: [4 N], not to be reused before
// the next barrier.
template <int N>
__device__ __forceinline__ void tile_sums(double (&v)[N], double* lds) {
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = wave_sum(v[k]);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < N; ++k) lds[4 * k + w] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k)
    v[k] = (lds[4 * k] + lds[4 * k + 1]) + (lds[4 * k + 2] + lds[4 * k + 3]);
}

// Final fold of one quantity over the tiles by one 256-thread workgroup:
// thread t sums part[t], part[t + 256], ... left to right from 0.0, then
// tile_sum (the oracle's final_combine).
// Eight loads are under way at a time (one after another, 4000 tiles took 5 us
// a fold): the zeros added past the end change no sum, which is never -0.
__device__ __forceinline__ double fold_strided(const double* part, int ntiles) {
  double acc = 0.0;
  for (int k = threadIdx.x; k < ntiles; k += 8 * PD_BLOCK) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = k + u * PD_BLOCK < ntiles ? part[k + u * PD_BLOCK] : 0.0;
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = acc + v[u];
  }
  return acc;
}
__device__ __forceinline__ double fold_partials(const double* part, int ntiles, double* lds4) {
  return tile_sum(fold_strided(part, ntiles), lds4);
}
// Two quantities at once, one exchange.
__device__ __forceinline__ void fold_pair(const double* part0, const double* part1, int ntiles,
                                          double* lds8, double& s0, double& s1) {
  double v[2] = {fold_strided(part0, ntiles), fold_strided(part1, ntiles)};
  tile_sums(v, lds8);
  s0 = v[0];
  s1 = v[1];
}

// The same over tiles t0 .. t0 + nt whose four slices' sums (wave_sum over 64
// rows each) are given instead: tile_sum's (w0 + w1) + (w2 + w3), slices past
// the last one summing to +0.
__device__ __forceinline__ double fold_slices(const double* slices, int nslices, int t0, int nt,
                                              double* lds4) {
  double acc = 0.0;
  for (int k = threadIdx.x; k < nt; k += PD_BLOCK) {
    const int s = 4 * (t0 + k);
    const double w0 = slices[s], w1 = s + 1 < nslices ? slices[s + 1] : 0.0;
    const double w2 = s + 2 < nslices ? slices[s + 2] : 0.0;
    const double w3 = s + 3 < nslices ? slices[s + 3] : 0.0;
    acc = acc + ((w0 + w1) + (w2 + w3));
  }
  return tile_sum(acc, lds4);
}
