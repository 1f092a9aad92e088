// pd_small.hip -- the FP64 step of systems that fit the chip at once (up to
// 256 slices): an assembly with L lanes per row, and one resident kernel
// that runs the whole CG solve.
//
// The general kernels give a row to a lane.  Below about 16,000 rows that
// leaves most SIMDs without a wave and makes every product as long as one
// lane's walk over its list (40 us at 8,000 rows), and an iteration costs
// four launches of about 4 us each.  Here a workgroup of 512 threads owns R
// = 512 / L rows, L = 8, 16 or 32 lanes per row:
//   * the lanes of a row evaluate its bonds side by side into LDS and a few
//     of them then add the terms in list order, so every sum has the order,
//     and the bits, of the one-lane walk;
//   * each lane keeps the 3x3 blocks of its slots on the chip for the whole
//     solve (with 8 lanes up to 15 of them, 13 in registers and two in LDS),
//     and the workgroup keeps p of its rows' neighbours in LDS: a product
//     multiplies from registers and LDS;
//   * the workgroups exchange z, p and the partial sums through global
//     memory without leaving the kernel.
// Steps before -> now: 288 rows 410 -> 114 us (assembly 13, solve 66), 8,000
// rows 755 -> 205 (assembly 93 -> 23; the solve, 149, was some 60 launches),
// 13,225 rows, Newmark, 504 -> 148 (26 and 96).  An iteration at 4,553 rows
// (143 workgroups): 9.1 us, of which the products and their sums 2.9, the
// waits for the two sums 3.9.
#include <math.h>

#include "pd_bond.h"
#include "pd_resident.h"

namespace pd {

namespace {

constexpr int kThreads = PD_SMALL_THREADS;

// Longest neighbour list of a unit that the solve keeps in LDS.  With 16 and
// 32 lanes no unit can have more (its rows, their bonds and row 0).
constexpr int small_union(int lanes) {
  return lanes == 8 ? PD_SMALL_UNION : kThreads / lanes * (PD_SMALL_MAX_BONDS + 1) + 1;
}

// Unit u of a solve with L lanes per row: slice u >> K, and of it the rows
// whose low K bits equal u's (K = log2(L / 8)), row i of the unit being row
// (i << K) + c of the slice.  The xor butterfly of a slice's wave sum pairs
// lanes 32, 16, .. 1 apart; a unit holds whole subtrees of its first 6 - K
// levels, and the remaining K levels join the slice's units.
template <int L>
struct Unit {
  static constexpr int R = kThreads / L;
  static constexpr int K = L == 8 ? 0 : L == 16 ? 1 : 2;
  static_assert(R << K == 64, "2^K units make a slice");
};

// Sum over the first R lanes (R = 16, 32 or 64), the butterfly's levels.
template <int R>
__device__ __forceinline__ double unit_sum(double v) {
  if constexpr (R > 32) v = xor_add<32>(v);
  if constexpr (R > 16) v = xor_add<16>(v);
  v = xor_add<8>(v);
  v = xor_add<4>(v);
  v = xor_add<2>(v);
  return xor_add<1>(v);
}

// Where unit u's partial lies in its row: eight to a 64-byte line, the lines
// 256 bytes apart so that the polls of all units spread over the memory
// channels.
__device__ __forceinline__ int small_slot(int u) { return (u >> 3) * 32 + (u & 7); }

// A partial that no unit has written yet: a signalling NaN, which no
// arithmetic returns (every partial is the result of an addition).
__device__ __forceinline__ double unset() {
  return __longlong_as_double((long long)0x7ff4deadbeef0001ull);
}
__device__ __forceinline__ bool is_unset(double v) {
  return (unsigned long long)__double_as_longlong(v) == 0x7ff4deadbeef0001ull;
}
__device__ __forceinline__ void put(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double get(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Every store of this wave has reached the point where all XCDs see it:
// stores that others read are agent-scope ones (written through), so their
// acknowledgement is all there is to wait for.  A release fence writes the
// whole L2 back on top, 1.5 to 2 us here.
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Fold of NV partial rows over tiles [t0, t0 + nt), nt <= 64 >> K, by one
// wave: fold_partials' tree.  The units' partials are read 64 at a time, one
// per lane (a lane per tile reading its units one after another asked for
// eight times the lines, 5 us a fold at 250 units); the lanes of a slice,
// then those of a tile join through xor levels (2^(K-1) .. 1 within the
// slice, then (w0 + w1) + (w2 + w3)), and tile t's sum moves to lane t.
// WAIT: the partials are written by running workgroups and awaited until all
// are set, the limit (ticks of the 100 MHz clock) has passed or another unit
// has given up (*aborted); then *late is raised.
template <int K, int NV, bool WAIT>
__device__ __forceinline__ void fold_units(const double* part, int64_t stride, int t0, int nt,
                                           int nslices, int lane, unsigned long long limit,
                                           const unsigned int* aborted, bool* late,
                                           double* out) {
  const int first = (t0 * 4) << K;
  const int nu = min(nt * 4, nslices - t0 * 4) << K;  // at most 256
  double v[NV][4];
  WaitLimit wait(limit);
  for (unsigned spin = 0;; ++spin) {
    bool ready = true;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        v[k][r] = r * 64 + lane < nu ? get(part + k * stride + small_slot(first + r * 64 + lane))
                                     : 0.0;
        if (WAIT) ready = ready && !is_unset(v[k][r]);
      }
    if (!WAIT || __all(ready)) break;
    if (WaitLimit::due(spin) &&
        (wait.over(spin, wall_clock64()) ||
         __hip_atomic_load(aborted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
      *late = true;
      break;
    }
  }
  constexpr int TPR = 16 >> K;  // tiles per 64 units
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double acc = 0.0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double x = v[k][r];
      if constexpr (K == 2) x = xor_add<1>(xor_add<2>(x));
      if constexpr (K == 1) x = xor_add<1>(x);
      x = xor_add<2 << K>(xor_add<1 << K>(x));
      const double y = __shfl(x, (lane % TPR) << (2 + K), 64);
      if (lane / TPR == r && lane < nt) acc = acc + y;
    }
    const double w = wave_sum(acc);
    out[k] = (w + 0.0) + (0.0 + 0.0);
  }
}

// chain_add (pd_device.h) over two lists of n terms side by side.
__device__ __forceinline__ void chain_add2(double (&acc)[2], const double* t0, const double* t1,
                                           int n) {
  double a0 = acc[0], a1 = acc[1];
  int e = 0;
  if (n >= 8) {
    double h0[8], h1[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      h0[u] = t0[u];
      h1[u] = t1[u];
    }
    for (; e + 16 <= n; e += 8) {
      double k0[8], k1[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        k0[u] = t0[e + 8 + u];
        k1[u] = t1[e + 8 + u];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        a0 += h0[u];
        a1 += h1[u];
        h0[u] = k0[u];
        h1[u] = k1[u];
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      a0 += h0[u];
      a1 += h1[u];
    }
    e += 8;
  }
  for (; e < n; ++e) {
    a0 += t0[e];
    a1 += t1[e];
  }
  acc[0] = a0;
  acc[1] = a1;
}

// The smallest and the largest over the L lanes of a row.
template <int L>
__device__ __forceinline__ void row_extremes(double& lo, double& hi) {
#pragma unroll
  for (int m = L / 2; m >= 1; m >>= 1) {
    const double l = __shfl_xor(lo, m, 64), h = __shfl_xor(hi, m, 64);
    lo = l < lo ? l : lo;
    hi = h > hi ? h : hi;
  }
}

// chain_add over t[0 .. n), n <= N wave-uniform, in steps of 16 terms with
// each term read 16 terms ahead (the terms past a list's end hold -0.0,
// which changes no sum).  An LDS read costs the same with one lane as with
// 64: a chain in three lanes of every wave took 32 cycles an addition, all
// eight waves reading; the chains of all rows side by side in one to three
// waves take about 10, the latency of the addition.
template <int N>
__device__ __forceinline__ double chain_wide(double acc, const double* t, int n) {
  static_assert(N % 16 == 0 || N % 8 == 0, "whole steps");
  double h[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) h[u] = u < N ? t[u] : -0.0;
#pragma unroll
  for (int e = 0; e < N; e += 16) {
    if (e >= n) break;  // uniform
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      if (e + u < N) acc += h[u];
      if (e + 16 + u < N) h[u] = t[e + 16 + u];
    }
  }
  return acc;
}

}  // namespace

// ---------------------------------------------------------------------------
// Assembly, L lanes per row: the sums of k_assemble<false, SHARED, true,
// false>, bit for bit.  A row's bonds are taken in chunks of 2 L slots, two
// per lane; each lane leaves its bonds' thirteen terms (force, Jacobian,
// first residual, stretch) in LDS and lane c then adds term c over the
// chunk in list order.  A chunk holding a breaking bond is redone after the
// row's list has been brought into its swap-remove order: the breaking
// bonds of the rest of the list are flagged in parallel, one lane walks the
// flags as the sequential pass walks the list, and the row's lanes apply
// the permutation.  Bound by latency: a chunk is a column load, a gather and
// 2 L additions in a row.  The stretch extremes are kept per lane: as chains of
// compares through LDS behind the sums they took a third of the kernel (288
// rows 21.8 -> 12.3 us, 8k 30.2 -> 22.3, 13k 37.3 -> 26.3).  Columns and records
// loaded a chunk ahead gained nothing (8k rows 13.1 us to the unit's end
// against 12.1, at 256 registers).
// ---------------------------------------------------------------------------
template <int L, bool SHARED>
__device__ __forceinline__ void small_assemble(const AsmArgs& a, const SmallArgs& g,
                                               double* lds) {
  constexpr int R = Unit<L>::R, K = Unit<L>::K;
  constexpr int CH = 2 * L, CP = CH + 1;  // slots per chunk and its padded stride
  constexpr int ROW = 13 * CP;            // LDS doubles per row
  constexpr int ROLES = 13;               // sums
  constexpr int NR = (ROLES + L - 1) / L;  // per lane
  static_assert(NR <= 2, "two chains side by side at most");
  const int unit = xcd_tile(blockIdx.x, gridDim.x);
  const int s = unit >> K;
  const int i = threadIdx.x / L, j = threadIdx.x % L;  // row of the unit, lane of the row
  const int pl = (i << K) + (unit & ((1 << K) - 1));
  const int p = s * 64 + pl;
  const bool vis = p < a.n && a.act[p] != PD_INVISIBLE;
  double* tr = lds + i * ROW;
  const int64_t base = a.slice_off[s];
  int top = vis ? a.top[p] : -1;
  pd_mat_dev mt = {1.0, 1.0, 1.0, 1.0};
  double4 pos_p = make_double4(0.0, 0.0, 0.0, 0.0);
  float stretch_f = 0.0f;
  if (vis) {
    mt = a.mat[a.body[p]];
    pos_p = a.x[p];
    stretch_f = (float)a.s[p];
  }
  int* __restrict__ col = a.col + base * 64 + pl;
  double* __restrict__ len = a.d0 + base * 64 + pl;
  const double hr = mt.horizon - mt.radius;
  const double yr = SHARED ? rcp_nr(mt.radius) : 0.0;
  bool short_len = false;
  double acc[2] = {0.0, 0.0};
  double smin = 0.0, smax = -INFINITY;  // of this lane's bonds

  // geometry, stretch and breaking test of slot k (k <= top)
  struct Bond {
    double4 u;
    double d0, e0, e1, e2, dij, yi, yd, dr;
    bool brk;
  };
  auto measure = [&](int q, double d0, Bond& b) {
    double4 xq;
    double sq;
    const dbl2v* r = (const dbl2v*)(a.arec + 8 * (int64_t)q);
    const dbl2v r0 = r[0], r1 = r[1], r2 = r[2], r3 = r[3];
    xq = make_double4(r0.x, r0.y, r1.x, 0.0);
    sq = r1.y;
    b.u = make_double4(r2.x, r2.y, r3.x, 0.0);
    b.d0 = d0;
    bond_dir<SHARED>(pos_p, xq, b.e0, b.e1, b.e2, b.dij, b.yi);
    b.yd = SHARED ? rcp_nr(d0) : 0.0;
    b.dr = (SHARED ? div_rcp(b.dij, d0, b.yd) : b.dij / d0) - 1.0;
    const float sq_f = (float)sq;
    b.brk = b.dr > (double)(stretch_f > sq_f ? stretch_f : sq_f);
  };
  const unsigned long long rowmask =
      (L == 64 ? ~0ull : ((1ull << L) - 1ull)) << ((threadIdx.x & 63) / L * L);
  int mt_top = top;  // longest list of the wave
#pragma unroll
  for (int m = 32; m >= L; m >>= 1) mt_top = max(mt_top, __shfl_xor(mt_top, m, 64));
  for (int c0 = 0; c0 <= mt_top; c0 += CH) {
    Bond b[2];
    bool rowbrk;
    for (int pass = 0;; ++pass) {
      int q[2];
      double l0[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int k = c0 + u * L + j;
        const bool in = k <= top;
        q[u] = in ? col[(int64_t)k * 64] : min(p, a.n - 1);
        l0[u] = in ? len[(int64_t)k * 64] : 1.0;
      }
      bool brk = false;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const bool in = c0 + u * L + j <= top;
        measure(q[u], l0[u], b[u]);
        if (in && SHARED) short_len = short_len || !((float)b[u].dij > small_len());
        brk = brk || (in && b[u].brk);
      }
      const unsigned long long any = __ballot(brk);
      rowbrk = pass == 0 && (any & rowmask) != 0;
      if (any == 0 || pass == 1) break;  // a redone chunk holds no breaking bond
      // flags of the row's slots from c0 on (128 slots at most)
      unsigned long long f0 = 0ull, f1 = 0ull;
      for (int k0 = c0; k0 <= mt_top; k0 += L) {
        const int k = k0 + j;
        const bool in = rowbrk && k <= top;
        bool bk = false;
        if (in) {
          Bond t;
          measure(col[(int64_t)k * 64], len[(int64_t)k * 64], t);
          if (SHARED) short_len = short_len || !((float)t.dij > small_len());
          bk = t.brk;
        }
        const unsigned long long bits =
            (__ballot(bk) & rowmask) >> ((threadIdx.x & 63) / L * L);
        if (k0 < 64)
          f0 |= bits << k0;  // k0 is a multiple of L, L divides 64
        else
          f1 |= bits << (k0 - 64);
      }
      // the row's list and the permutation in LDS (the chunk's terms are not
      // written yet, the previous chunk's have been added)
      double* dS = tr;                       // [128]
      int* cS = (int*)(tr + 128);            // [128]
      unsigned char* perm = (unsigned char*)(tr + 192);  // [128]
      static_assert(192 + 16 <= ROW, "list, lengths and permutation fit a row's terms");
      wave_fence();
      if (rowbrk)
        for (int k = c0 + j; k <= top; k += L) {
          dS[k] = len[(int64_t)k * 64];
          cS[k] = col[(int64_t)k * 64];
          perm[k] = (unsigned char)k;
        }
      wave_fence();
      int ntop = top;
      if (rowbrk) {  // every lane of the row walks alike; lane 0 writes
        while (true) {
          // the first flagged slot at or below ntop
          const int w = f0 ? __ffsll((long long)f0) - 1 : f1 ? 64 + __ffsll((long long)f1) - 1 : 128;
          if (w > ntop) break;
          const bool tb = ntop < 64 ? (f0 >> ntop) & 1ull : (f1 >> (ntop - 64)) & 1ull;
          // swap slots w and ntop; the flag of ntop moves to w, ntop is dead
          if (j == 0) {
            const unsigned char t = perm[w];
            perm[w] = perm[ntop];
            perm[ntop] = t;
          }
          if (!tb) {
            if (w < 64)
              f0 &= ~(1ull << w);
            else
              f1 &= ~(1ull << (w - 64));
          }
          if (ntop < 64)
            f0 &= ~(1ull << ntop);
          else
            f1 &= ~(1ull << (ntop - 64));
          if (tb && w != ntop) {  // w holds a breaking bond again
            if (w < 64)
              f0 |= 1ull << w;
            else
              f1 |= 1ull << (w - 64);
          }
          --ntop;
        }
      }
      wave_fence();
      if (rowbrk) {
        for (int k = c0 + j; k <= top; k += L) {
          const int o = perm[k];
          if (o != k) {
            col[(int64_t)k * 64] = cS[o];
            len[(int64_t)k * 64] = dS[o];
          }
        }
        top = ntop;
      }
      __threadfence_block();  // the row's other lanes read the list back
      wave_fence();
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const Bond& t = b[u];
      double vscale = 1.0;
      if (t.d0 > hr)
        vscale = 0.5 + (SHARED ? div_rcp((mt.horizon - t.d0) / 2.0, mt.radius, yr)
                               : (mt.horizon - t.d0) / 2.0 / mt.radius);
      const double kk = t.dr * vscale;
      double F00, F01, F02, F11, F12, F22;
      const double sc = SHARED ? div_rcp(mt.c_bond, t.d0, t.yd) : mt.c_bond / t.d0;
      bond_jac_sc<SHARED, false>(t.e0, t.e1, t.e2, t.dij, t.yi, t.d0, sc, F00, F01, F02, F11,
                                 F12, F22);
      const double b00 = (F00 * -1.0) * a.dt2, b01 = (F01 * -1.0) * a.dt2,
                   b02 = (F02 * -1.0) * a.dt2, b11 = (F11 * -1.0) * a.dt2,
                   b12 = (F12 * -1.0) * a.dt2, b22 = (F22 * -1.0) * a.dt2;
      double* o = tr + u * L + j;
      o[0 * CP] = kk * t.e0;
      o[1 * CP] = kk * t.e1;
      o[2 * CP] = kk * t.e2;
      o[3 * CP] = F00;
      o[4 * CP] = F01;
      o[5 * CP] = F02;
      o[6 * CP] = F11;
      o[7 * CP] = F12;
      o[8 * CP] = F22;
      o[9 * CP] = b00 * t.u.x + b01 * t.u.y + b02 * t.u.z;
      o[10 * CP] = b01 * t.u.x + b11 * t.u.y + b12 * t.u.z;
      o[11 * CP] = b02 * t.u.x + b12 * t.u.y + b22 * t.u.z;
      o[12 * CP] = t.dr;
      if (c0 + u * L + j <= top) {
        smin = t.dr < smin ? t.dr : smin;
        smax = t.dr > smax ? t.dr : smax;
      }
    }
    wave_fence();
    const int m = min(CH, top + 1 - c0);
    // lane j adds terms j and j + L (lanes past the last repeat it)
    if constexpr (NR == 2)
      chain_add2(acc, tr + j * CP, tr + min(j + L, ROLES - 1) * CP, m);
    else
      acc[0] = chain_add(acc[0], tr + min(j, ROLES - 1) * CP, m);
    wave_fence();
  }
  // the row's sums to the unit's owner lanes (the first R threads)
  __syncthreads();
  double* sum = lds;  // [R][16]
#pragma unroll
  for (int k = 0; k < NR; ++k)
    if (j + k * L < ROLES) sum[i * 16 + j + k * L] = acc[k];
  row_extremes<L>(smin, smax);
  if (j == 0) {
    sum[i * 16 + 13] = smin;
    sum[i * 16 + 14] = smax;
  }
  int* tops = (int*)(lds + R * 16);  // [R]
  if (j == 0) tops[i] = top;
  const bool zany = __any(short_len);
  if (SHARED && zany && (threadIdx.x & 63) == 0) atomicOr(&a.counters->range_bad, 2u);
  __syncthreads();
  if (threadIdx.x >= 64) return;
  // one lane per row: k_assemble's end of a row
  const int ri = threadIdx.x;
  const int rl = (ri << K) + (unit & ((1 << K) - 1));
  const int rp = s * 64 + rl;
  double t_rr = 0.0, t_rz = 0.0, t_bb = 0.0;
  unsigned long long broken = 0, live = 0;
  if (ri < R && rp < a.n) {
    double* ex = g.ex + 6 * (int64_t)rp;
    if (a.act[rp] != PD_INVISIBLE) {
      const pd_mat_dev rm = a.mat[a.body[rp]];
      const double* q = sum + ri * 16;
      const int rtop = tops[ri];
      const double d00 = q[3] * a.dt2 + rm.mass;
      const double d01 = q[4] * a.dt2 + 0.0;
      const double d02 = q[5] * a.dt2 + 0.0;
      const double d11 = q[6] * a.dt2 + rm.mass;
      const double d12 = q[7] * a.dt2 + 0.0;
      const double d22 = q[8] * a.dt2 + rm.mass;
      double* dg = a.diag + (int64_t)s * 384 + rl;
      dg[0] = d00;
      dg[64] = d01;
      dg[128] = d02;
      dg[192] = d11;
      dg[256] = d12;
      dg[320] = d22;
      const double c00 = d11 * d22 - d12 * d12;
      const double c01 = d02 * d12 - d01 * d22;
      const double c02 = d01 * d12 - d02 * d11;
      const double c11 = d00 * d22 - d02 * d02;
      const double c12 = d01 * d02 - d00 * d12;
      const double c22 = d00 * d11 - d01 * d01;
      const double det = (d00 * c00 + d01 * c01) + d02 * c02;
      const double id = 1.0 / det;
      const double m0 = c00 * id, m1 = c01 * id, m2 = c02 * id, m3 = c11 * id, m4 = c12 * id,
                   m5 = c22 * id;
      double* mo = a.minv + (int64_t)s * 384 + rl;
      mo[0] = m0;
      mo[64] = m1;
      mo[128] = m2;
      mo[192] = m3;
      mo[256] = m4;
      mo[320] = m5;
      double f0 = q[0] * rm.c_bond, f1 = q[1] * rm.c_bond, f2 = q[2] * rm.c_bond;
      const double ss0 = (10.0 - 9.0 * a.clock) * a.s00[rp];
      a.s_new[rp] = ss0 - 0.25 * q[13];
      f1 -= (a.clock * a.gravity * rm.mass);
      if (a.contact) {
        const double4 c = a.fc[rp];
        const double l = sqrt(c.x * c.x + c.y * c.y + c.z * c.z);
        if (l > 1e-10) {
          f0 += c.x;
          f1 += c.y;
          f2 += c.z;
        }
      }
      a.f[rp] = make_double4(f0, f1, f2, 0.0);
      const double4 vp = a.v[rp];
      double4 bo;
      if (a.integrator == 1) {
        const double hdt = 0.5 * a.dt;
        bo.x = a.dt * (rm.mass * vp.x + hdt * f0);
        bo.y = a.dt * (rm.mass * vp.y + hdt * f1);
        bo.z = a.dt * (rm.mass * vp.z + hdt * f2);
      } else {
        bo.x = rm.mass * vp.x + a.dt * f0;
        bo.y = rm.mass * vp.y + a.dt * f1;
        bo.z = rm.mass * vp.z + a.dt * f2;
      }
      bo.w = 0.0;
      a.b[rp] = bo;
      const double4 xp = a.xs[rp];
      const double y0 = (d00 * xp.x + d01 * xp.y + d02 * xp.z) + q[9];
      const double y1 = (d01 * xp.x + d11 * xp.y + d12 * xp.z) + q[10];
      const double y2 = (d02 * xp.x + d12 * xp.y + d22 * xp.z) + q[11];
      const bool fr = a.bc[rp] == 0;
      const double r0 = fr ? bo.x - y0 : 0.0;
      const double r1 = fr ? bo.y - y1 : 0.0;
      const double r2 = fr ? bo.z - y2 : 0.0;
      const double sb0 = fr ? bo.x : 0.0, sb1 = fr ? bo.y : 0.0, sb2 = fr ? bo.z : 0.0;
      t_rr = (r0 * r0 + r1 * r1) + r2 * r2;
      t_bb = (sb0 * sb0 + sb1 * sb1) + sb2 * sb2;
      double z0 = r0, z1 = r1, z2 = r2;
      if (a.pc) {
        z0 = m0 * r0 + m1 * r1 + m2 * r2;
        z1 = m1 * r0 + m3 * r1 + m4 * r2;
        z2 = m2 * r0 + m4 * r1 + m5 * r2;
      }
      a.r64[rp] = make_double4(r0, r1, r2, 0.0);
      ex[0] = z0;
      ex[1] = z1;
      ex[2] = z2;
      t_rz = (r0 * z0 + r1 * z1) + r2 * z2;
      // the row's list before this step ended at its owner's a.top
      const int was = a.top[rp];
      if (rtop != was) {
        a.top[rp] = rtop;
        broken = (unsigned long long)(was - rtop);
      }
      live = (unsigned long long)(rtop + 1);
      if (a.bond_stats)
        a.bond_stats[rp] = make_float2(rtop >= 0 ? (float)(q[12] / (rtop + 1)) : 0.0f,
                                       rtop >= 0 ? (float)q[14] : 0.0f);
    } else {
      a.r64[rp] = make_double4(0.0, 0.0, 0.0, 0.0);
      ex[0] = 0.0;
      ex[1] = 0.0;
      ex[2] = 0.0;
    }
  }
  const double v0 = unit_sum<R>(t_rz), v1 = unit_sum<R>(t_rr), v2 = unit_sum<R>(t_bb);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    broken += __shfl_xor(broken, m, 64);
    live += __shfl_xor(live, m, 64);
  }
  if (threadIdx.x == 0) {
    const int at = small_slot(unit);
    g.start[at] = v0;
    g.start[PD_SMALL_ROW + at] = v1;
    g.start[2 * PD_SMALL_ROW + at] = v2;
#pragma unroll
    for (int k = 0; k < 6; ++k) g.part[k * PD_SMALL_ROW + at] = unset();
    if (broken) atomicAdd(&a.counters->broken, broken);
    if (live) atomicAdd(&a.counters->live, live);
    if (unit == 0) *g.aborted = 0u;
  }
}

template <int L>
__global__ __launch_bounds__(kThreads) void k_small_assemble(AsmArgs a, SmallArgs g) {
  __shared__ double lds[Unit<L>::R * 13 * (2 * L + 1)];
  if ((a.counters->range_bad & 1u) == 0)  // uniform over the grid
    small_assemble<L, true>(a, g, lds);
  else
    small_assemble<L, false>(a, g, lds);
}

// ---------------------------------------------------------------------------
// The CG solve of a step in one launch, every workgroup resident: CUSP's
// loop as the general kernels run it (k_cg_spmv, k_cg_update, k_cg_beta,
// k_cg_dir), the same sums in the same order.
//
// An iteration: the workgroup forms p = z + beta p of its rows' neighbours
// in LDS, every lane multiplies its blocks by it and leaves the terms in
// LDS, and the first wave adds them in list order on top of the diagonal
// terms.  Its first R lanes then own a row each: <y, p>, and
// once every unit's partial is there alpha, x, r, z; once <r, z> and <r, r>
// are there, beta and the monitor test.  A unit's partial doubles as its
// arrival: partials are awaited until they are set, and those of the
// phase before are unset again once the next phase's are complete (all
// units have read them by then).  z and p go through global memory, by
// agent-scope stores that are awaited ahead of the partial and an agent
// acquire after the wait, by one wave per workgroup (fences in all eight
// took 30 to 60 us per round; in one they are not seen).
//
// Every wait ends: after g.spin_ticks of the 100 MHz clock, counted anew in
// each wait, a workgroup raises *g.aborted and leaves (0 ticks: before the
// first iteration, whatever the others do).  The position update behind it
// then does nothing, and the host puts the start values back (the assembly
// record holds them) and solves with the general kernels.
// ---------------------------------------------------------------------------
// M slots per lane, the blocks of the first MR in registers and of the rest
// in LDS; MC slots per chunk.
template <int L, int M, int MR, int MC>
__global__ __launch_bounds__(kThreads) void k_small_solve(CgArgs a, SmallArgs g) {
  constexpr int R = Unit<L>::R, K = Unit<L>::K;
  constexpr int CH = MC * L, CP = CH + 3;  // slots per chunk, padded stride
  __shared__ __attribute__((aligned(16))) double T[R * 3 * CP];  // terms
  __shared__ double Y[3 * R];
  __shared__ double Di[6 * R];  // the rows' diagonal blocks
  __shared__ int longest;
  __shared__ int own_l[R];  // each row's p in V
  // the owners' x and r wait in LDS where the blocks leave no registers
  constexpr bool kStateLds = L == 8;
  __shared__ double Sl[kStateLds ? 6 * R : 1];
  __shared__ double Mi[6 * R];  // and their inverses
  // the unit's neighbours: the rows its blocks touch and its own, ascending
  constexpr int UC = small_union(L);
  __shared__ unsigned short list[UC];
  __shared__ double V[3 * UC];  // their p of this iteration
  __shared__ dbl2v Bl[M > MR ? (M - MR) * 3 * kThreads : 1];
  __shared__ double ctl[2];     // beta, and whether the loop goes on
  const int unit = xcd_tile(blockIdx.x, gridDim.x);
  const int s = unit >> K, cl = unit & ((1 << K) - 1);
  const int i = threadIdx.x / L, j = threadIdx.x % L;
  const int pl = (i << K) + cl;
  const int p = s * 64 + pl;
  const bool row = p < a.A.n;
  const int top = row ? a.A.top[p] : -1;
  const int spec = spec_of(a.batch, s >> 2);
  int t0, nt;
  spec_range_of(a.batch, spec, (a.A.n + PD_BLOCK - 1) / PD_BLOCK, t0, nt);
  if (unit == 0 && threadIdx.x == 0) *g.h_cnt = *g.counters;
  // a tile before the first specimen, between two or behind the last: its rows
  // are invisible and nobody awaits its sums, so it may not await others' (they
  // are unset again as soon as the specimen's own units have read them)
  if ((s >> 2) < t0 || (s >> 2) >= t0 + nt) return;
  // the slots' blocks (past the list's end anything: nothing adds them)
  int q[M];
  double B[MR][6];
  {
    const int64_t base = a.A.slice_off[s];
    const int* __restrict__ cp = a.A.col + base * 64 + pl;
    const double* __restrict__ lp = a.A.d0 + base * 64 + pl;
    const int pc = row ? p : 0;
    const double4 pos_p = a.A.pos[pc];
    const double cb = a.A.mat[a.A.body[pc]].c_bond;
    const double dt2 = a.A.dt2;
    const bool shared = *a.A.range_bad == 0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int k = m * L + j;
      q[m] = k <= top ? ntl(cp + (int64_t)k * 64) : -1;
    }
    // groups of GS slots: their loads go out together
    constexpr int GS = 4;
#pragma unroll
    for (int m0 = 0; m0 < M; m0 += GS) {
      double l0[GS];
      double4 xq[GS];
#pragma unroll
      for (int u = 0; u < GS; ++u) {
        if (m0 + u >= M) break;
        const int m = m0 + u;
        l0[u] = q[m] >= 0 ? ntl(lp + (int64_t)(m * L + j) * 64) : 1.0;
        xq[u] = a.A.pos[q[m] >= 0 ? q[m] : pc];
      }
#pragma unroll
      for (int u = 0; u < GS; ++u) {
        if (m0 + u >= M) break;
        const int m = m0 + u;
        double e0, e1, e2, dij, yi, F00, F01, F02, F11, F12, F22;
        if (shared) {
          bond_dir<true, true>(pos_p, xq[u], e0, e1, e2, dij, yi);
          bond_jac<true>(e0, e1, e2, dij, yi, l0[u], cb, F00, F01, F02, F11, F12, F22);
        } else {
          bond_dir(pos_p, xq[u], e0, e1, e2, dij, yi);
          bond_jac(e0, e1, e2, dij, yi, l0[u], cb, F00, F01, F02, F11, F12, F22);
        }
        const double b0 = (F00 * -1.0) * dt2, b1 = (F01 * -1.0) * dt2, b2 = (F02 * -1.0) * dt2,
                     b3 = (F11 * -1.0) * dt2, b4 = (F12 * -1.0) * dt2, b5 = (F22 * -1.0) * dt2;
        if (m < MR) {
          B[m < MR ? m : 0][0] = b0;
          B[m < MR ? m : 0][1] = b1;
          B[m < MR ? m : 0][2] = b2;
          B[m < MR ? m : 0][3] = b3;
          B[m < MR ? m : 0][4] = b4;
          B[m < MR ? m : 0][5] = b5;
        } else {
          dbl2v* o = Bl + (m - MR) * 3 * kThreads + threadIdx.x;
          o[0] = dbl2v{b0, b1};
          o[kThreads] = dbl2v{b2, b3};
          o[2 * kThreads] = dbl2v{b4, b5};
        }
        if (q[m] < 0)
          q[m] = pc;  // past the list's end: a gather in bounds, its term unused
        else if (a.vals)
          store_block(a.vals, base + m * L + j, pl, b0, b1, b2, b3, b4, b5);
      }
    }
  }
  // the union of the gathered rows as a bitmap, its ranks the local indices.
  // The rows are marked by a byte each, stored plainly: a bit each, by LDS
  // atomics, had most of a wave's lanes queue at a few words (the neighbours
  // of neighbouring rows): 24 thousand cycles of a solve's set-up at 13k rows
  // against 12.
  int own_at, nlist;
  unsigned int at2[(M + 1) / 2];  // slots' places in V, two to a word
  static_assert(3 * small_union(L) <= 65536, "16-bit places");
  {
    typedef unsigned int u4v __attribute__((ext_vector_type(4)));
    typedef unsigned int u2v __attribute__((ext_vector_type(2)));
    u4v* marks = (u4v*)T;                                // [2 kThreads]: 16,384 rows
    u2v* words = (u2v*)(marks + 2 * kThreads);           // [kThreads] bits, ones before the word
    unsigned int* wsum = (unsigned int*)(words + kThreads);  // [kThreads / 64]
    static_assert(sizeof(T) >= 2 * kThreads * 16 + kThreads * 8 + kThreads / 64 * 4, "scratch");
    static_assert(PD_SMALL_UNITS * 64 <= kThreads * 32, "a byte per row");
    const int t = threadIdx.x, wl = t & 63;
    const int pc = row ? p : 0;
    marks[t] = u4v{0u, 0u, 0u, 0u};
    marks[kThreads + t] = u4v{0u, 0u, 0u, 0u};
    if (t == 0) longest = 0;
    __syncthreads();
    unsigned char* mark = (unsigned char*)marks;
#pragma unroll
    for (int m = 0; m < M; ++m) mark[q[m]] = 1;
    if (j == 0) mark[pc] = 1;
    __syncthreads();
    unsigned int mine = 0u;  // rows 32 t ..
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const u4v v = marks[2 * t + h];
#pragma unroll
      for (int k = 0; k < 4; ++k)  // four bytes of 0 or 1 to four bits
        mine |= ((v[k] * 0x01020408u) >> 24 & 0xfu) << (16 * h + 4 * k);
    }
    int incl = __popc(mine);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(incl, d, 64);
      if (wl >= d) incl += v;
    }
    if (wl == 63) wsum[t >> 6] = incl;
    __syncthreads();
    int before = 0;
    nlist = 0;
#pragma unroll
    for (int k = 0; k < kThreads / 64; ++k) {
      if (k < (t >> 6)) before += wsum[k];
      nlist += wsum[k];
    }
    const int ex0 = before + incl - __popc(mine);
    words[t] = u2v{mine, (unsigned int)ex0};
    unsigned int left = mine;
    for (int k = ex0; left; ++k) {
      if (k < UC) list[k] = (unsigned short)(t * 32 + __ffs((int)left) - 1);
      left &= left - 1;
    }
    __syncthreads();
    auto local = [&](int r) {
      const u2v w = words[r >> 5];
      return 3 * (int)(w.y + __popc(w.x & ((1u << (r & 31)) - 1u)));
    };
#pragma unroll
    for (int m = 0; m < M; m += 2) {
      unsigned int h = (unsigned int)local(q[m]);
      if (m + 1 < M) h |= (unsigned int)local(q[m + 1]) << 16;
      at2[m / 2] = h;
    }
    own_at = local(pc);
    __syncthreads();
  }
  nlist = min(nlist, UC);  // the host found that no unit has more (k_small_union)
  if (j == 0) {
    own_l[i] = own_at;
    atomicMax(&longest, top + 1);
  }
  // the first R threads own a row each
  const int ol = (threadIdx.x << K) + cl;
  const int op = s * 64 + ol;
  const bool own = threadIdx.x < R && op < a.A.n;
  double x0 = 0.0, x1 = 0.0, x2 = 0.0, r0 = 0.0, r1 = 0.0, r2 = 0.0;
  bool fr = false;
  if (own) {
    const double4 xx = a.x[op], rr = a.r[op];
    x0 = xx.x;
    x1 = xx.y;
    x2 = xx.z;
    r0 = rr.x;
    r1 = rr.y;
    r2 = rr.z;
    fr = a.bc[op] == 0;
    const int64_t blk = (int64_t)s * 384 + ol;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      Di[c * R + threadIdx.x] = a.A.diag[blk + c * 64];
      if (a.precond) Mi[c * R + threadIdx.x] = a.minv[blk + c * 64];
    }
  }
  auto state = [&](bool load) {
    if constexpr (kStateLds) {
      double* o = Sl + threadIdx.x;
      double* v[6] = {&x0, &x1, &x2, &r0, &r1, &r2};
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        if (load)
          *v[k] = o[k * R];
        else
          o[k * R] = *v[k];
      }
    }
  };
  if (own) state(false);
  const int lane = threadIdx.x & 63;
  const bool lead = threadIdx.x < 64;  // the wave of the owners
  bool late = false;
  double rz = 0.0, rr = 0.0, tol = 0.0, bnorm = 0.0, rnorm = 0.0, alpha = 0.0, beta = 0.0,
         yp = 0.0;
  int iter = 0;
  bool done = false, conv = false;
  if (lead) {
    double v[3];
    fold_units<K, 3, false>(g.start, PD_SMALL_ROW, t0, nt, g.nslices, lane, 0, nullptr, &late, v);
    rz = v[0];
    rr = v[1];
    const double bb = v[2];
    bnorm = sqrt(bb);
    tol = g.rtol * bnorm;
    rnorm = sqrt(rr);
    if (rnorm <= tol) {
      done = true;
      conv = true;
    } else if (g.max_iter <= 0) {
      done = true;
    }
    late = g.spin_ticks == 0;  // no wait at all
    if (threadIdx.x == 0) {
      ctl[0] = 0.0;
      ctl[1] = done || late ? 0.0 : 1.0;
    }
  }
  __syncthreads();
  const int64_t exn = 6 * (int64_t)a.A.n;
  const int most = __builtin_amdgcn_readfirstlane(longest);  // slots in use
  const int chain_c = threadIdx.x / R, chain_row = threadIdx.x % R;
  const int at = small_slot(unit);
  constexpr int PR = PD_SMALL_ROW;
  double* P_yp = g.part;
  double* P_rz = g.part + 2 * PR;  // and <r, r> two rows on
  for (int it = 0; ctl[1] != 0.0; ++it) {
    const double bt = ctl[0];
    const double* ex = g.ex + (it & 1 ? exn : 0);
    // p = z + beta p of the neighbours (z in the first iteration), once each
#pragma unroll 4
    for (int k = threadIdx.x; k < nlist; k += kThreads) {
      const dbl2v* e = (const dbl2v*)(ex + 6 * (int64_t)list[k]);
      const dbl2v ea = e[0], eb = e[1], ec = e[2];
      double v0 = ea.x, v1 = ea.y, v2 = eb.x;
      if (it > 0) {
        v0 = v0 + bt * eb.y;
        v1 = v1 + bt * ec.x;
        v2 = v2 + bt * ec.y;
      }
      V[3 * k] = v0;
      V[3 * k + 1] = v1;
      V[3 * k + 2] = v2;
    }
    __syncthreads();
    double acc = 0.0;
    if (threadIdx.x < 3 * R) {  // the diagonal term comes first
      const double* v = V + own_l[chain_row];
      const double* d = Di + chain_row;
      acc = d[chain_c * R] * v[0] + d[(chain_c == 0 ? 1 : chain_c + 2) * R] * v[1] +
            d[(chain_c == 0 ? 2 : chain_c + 3) * R] * v[2];
    }
#pragma unroll
    for (int m0 = 0; m0 < M; m0 += MC) {
#pragma unroll
      for (int m = m0; m < m0 + MC; ++m) {
        if (m >= M) {  // the last chunk's slots that no list reaches
          double* o = T + i * 3 * CP + (m - m0) * L + j;
          o[0] = -0.0;
          o[CP] = -0.0;
          o[2 * CP] = -0.0;
          continue;
        }
        double u0, u1, u2;
        const double* v = V + (m & 1 ? at2[m / 2] >> 16 : at2[m / 2] & 0xffffu);
        const double4 v4 = make_double4(v[0], v[1], v[2], 0.0);
        if (m < MR) {
          const double* k = B[m < MR ? m : 0];
          blk6(k[0], k[1], k[2], k[3], k[4], k[5], v4, u0, u1, u2);
        } else {
          const dbl2v* k = Bl + (m - MR) * 3 * kThreads + threadIdx.x;
          const dbl2v ka = k[0], kb = k[kThreads], kc = k[2 * kThreads];
          blk6(ka.x, ka.y, kb.x, kb.y, kc.x, kc.y, v4, u0, u1, u2);
        }
        const bool in = m * L + j <= top;
        double* o = T + i * 3 * CP + (m - m0) * L + j;
        o[0] = in ? u0 : -0.0;
        o[CP] = in ? u1 : -0.0;
        o[2 * CP] = in ? u2 : -0.0;
      }
      __syncthreads();
      if (threadIdx.x < 3 * R) {  // a lane per row and component
        const int n = most - m0 * L;
        if (n > 0) acc = chain_wide<CH>(acc, T + (chain_row * 3 + chain_c) * CP, n);
      }
      if (m0 + MC < M) __syncthreads();
    }
    if (threadIdx.x < 3 * R) Y[threadIdx.x] = acc;
    __syncthreads();
    if (lead) {
      const int b = it & 1;
      double t_yp = 0.0, y0 = 0.0, y1 = 0.0, y2 = 0.0, p0 = 0.0, p1 = 0.0, p2 = 0.0;
      if (own) {
        y0 = Y[threadIdx.x];
        y1 = Y[R + threadIdx.x];
        y2 = Y[2 * R + threadIdx.x];
        const double* v = V + own_l[threadIdx.x];
        p0 = v[0];
        p1 = v[1];
        p2 = v[2];
        t_yp = (y0 * p0 + y1 * p1) + y2 * p2;
      }
      const double vy = unit_sum<R>(t_yp);
      if (lane == 0) put(P_yp + b * PR + at, vy);
      // the record that the next iteration gathers
      double* e = g.ex + (b ? 0 : exn) + 6 * (int64_t)op;
      if (own) {
        put(e + 3, p0);
        put(e + 4, p1);
        put(e + 5, p2);
      }
      fold_units<K, 1, true>(P_yp + b * PR, 0, t0, nt, g.nslices, lane, g.spin_ticks, g.aborted,
                             &late, &yp);
      alpha = rz / yp;
      double t_rz = 0.0, t_rr = 0.0;
      if (own) {
        state(true);
        x0 = alpha * p0 + x0;
        x1 = alpha * p1 + x1;
        x2 = alpha * p2 + x2;
        if (fr) {
          const double na = -alpha;
          r0 = na * y0 + r0;
          r1 = na * y1 + r1;
          r2 = na * y2 + r2;
        }
        double z0 = r0, z1 = r1, z2 = r2;
        if (a.precond) {
          const double* m = Mi + threadIdx.x;
          const double m00 = m[0], m01 = m[R], m02 = m[2 * R], m11 = m[3 * R], m12 = m[4 * R],
                       m22 = m[5 * R];
          z0 = m00 * r0 + m01 * r1 + m02 * r2;
          z1 = m01 * r0 + m11 * r1 + m12 * r2;
          z2 = m02 * r0 + m12 * r1 + m22 * r2;
        }
        put(e, z0);
        put(e + 1, z1);
        put(e + 2, z2);
        t_rz = (r0 * z0 + r1 * z1) + r2 * z2;
        t_rr = (r0 * r0 + r1 * r1) + r2 * r2;
        state(false);
      }
      const double vz = unit_sum<R>(t_rz), vr = unit_sum<R>(t_rr);
      if (lane == 0 && it > 0) {  // all units have read the previous <r, z>
        put(P_rz + (b ^ 1) * PR + at, unset());
        put(P_rz + (2 + (b ^ 1)) * PR + at, unset());
      }
      stores_done();
      if (lane == 0) {
        put(P_rz + b * PR + at, vz);
        put(P_rz + (2 + b) * PR + at, vr);
      }
      double sums[2];
      fold_units<K, 2, true>(P_rz + b * PR, 2 * PR, t0, nt, g.nslices, lane, g.spin_ticks,
                             g.aborted, &late, sums);
      const double nrz = sums[0];
      rr = sums[1];
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      // all units have read this iteration's <y, p>
      if (lane == 0) put(P_yp + b * PR + at, unset());
      beta = nrz / rz;
      rz = nrz;
      ++iter;
      rnorm = sqrt(rr);
      if (rnorm <= tol) {
        done = true;
        conv = true;
      } else if (iter >= g.max_iter) {
        done = true;
      }
      if (threadIdx.x == 0) {
        ctl[0] = beta;
        ctl[1] = done || late ? 0.0 : 1.0;
      }
    }
    __syncthreads();
  }
  if (!lead) return;
  if (late) {  // uniform over the wave
    if (threadIdx.x == 0) {
      atomicOr(g.aborted, 1u);
      *g.h_aborted = 1u;
    }
    return;
  }
  if (own) {
    state(true);
    a.x[op] = make_double4(x0, x1, x2, 0.0);
  }
  if (threadIdx.x == 0 && s == 4 * t0 && cl == 0) {  // the specimen's first unit
    pd_cg_state* st = g.h_st + spec;
    st->rz = rz;
    st->yp = yp;
    st->alpha = alpha;
    st->beta = beta;
    st->rr = rr;
    st->bnorm = bnorm;
    st->tol = tol;
    st->rnorm = rnorm;
    st->rtol = g.rtol;
    st->iter = iter;
    st->done = 1;
    st->converged = conv ? 1 : 0;
    st->max_iter = g.max_iter;
    st->upd_it = iter - 1;
  }
}

// The longest of the units' neighbour lists, over all the slots a list may
// hold (its capacity): with 8 lanes per row it may exceed what LDS holds.
template <int L>
__global__ __launch_bounds__(kThreads) void k_small_union(int n, const int64_t* slice_off,
                                                          const int32_t* cap, const int32_t* col,
                                                          int* longest) {
  constexpr int K = Unit<L>::K;
  __shared__ unsigned int bits[kThreads];
  __shared__ int total;
  const int unit = blockIdx.x, s = unit >> K;
  const int pl = ((threadIdx.x / L) << K) + (unit & ((1 << K) - 1)), p = s * 64 + pl;
  bits[threadIdx.x] = 0u;
  if (threadIdx.x == 0) total = 0;
  __syncthreads();
  if (p < n) {
    const int* c = col + slice_off[s] * 64 + pl;
    for (int k = threadIdx.x % L; k < cap[p]; k += L) {
      const int q = c[(int64_t)k * 64];
      atomicOr(bits + (q >> 5), 1u << (q & 31));
    }
    atomicOr(bits + (p >> 5), 1u << (p & 31));
  }
  __syncthreads();
  atomicAdd(&total, __popc(bits[threadIdx.x]));
  __syncthreads();
  if (threadIdx.x == 0) atomicMax(longest, total + 1);  // row 0 stands in for absent ones
}

void launch_small_union(int32_t n, int32_t nslices, const int64_t* slice_off, const int32_t* cap,
                        const int32_t* col, int* longest, hipStream_t s) {
  hipLaunchKernelGGL(k_small_union<8>, dim3(nslices), dim3(kThreads), 0, s, n, slice_off, cap,
                     col, longest);
}

// the solve's start values back into x, after a solve that gave up
__global__ __launch_bounds__(PD_BLOCK) void k_small_undo(int n, const double* arec, double4* x) {
  const int p = blockIdx.x * PD_BLOCK + threadIdx.x;
  if (p >= n) return;
  const double* r = arec + 8 * (int64_t)p;
  x[p] = make_double4(r[4], r[5], r[6], 0.0);
}

void launch_small_undo(int32_t n, const double* arec, double4* x, hipStream_t s) {
  const int nb = (n + PD_BLOCK - 1) / PD_BLOCK;
  if (nb) hipLaunchKernelGGL(k_small_undo, dim3(nb), dim3(PD_BLOCK), 0, s, n, arec, x);
}

void launch_small_assemble(int lanes, const AsmArgs& a, const SmallArgs& g, hipStream_t s) {
  const dim3 grid(g.units), block(kThreads);
  switch (lanes) {
    case 8: hipLaunchKernelGGL(k_small_assemble<8>, grid, block, 0, s, a, g); break;
    case 16: hipLaunchKernelGGL(k_small_assemble<16>, grid, block, 0, s, a, g); break;
    default: hipLaunchKernelGGL(k_small_assemble<32>, grid, block, 0, s, a, g);
  }
}

// slots per lane (L * M >= PD_SMALL_MAX_BONDS), those in registers, slots
// per chunk (its gathers are in flight together).  With 8 lanes not all
// fifteen fit the 256 registers beside a chunk's gathers (all in registers 32
// spill, fourteen 17), and LDS has room for two slots beside the rest (163,040
// of 163,840 bytes), so thirteen stay in registers (4 spill).
#define SOLVE8 k_small_solve<8, 15, 13, 4>
#define SOLVE16 k_small_solve<16, 8, 8, 4>
#define SOLVE32 k_small_solve<32, 4, 4, 4>
static_assert(8 * 15 >= PD_SMALL_MAX_BONDS && 16 * 8 >= PD_SMALL_MAX_BONDS &&
                  32 * 4 >= PD_SMALL_MAX_BONDS,
              "a row's blocks fit its lanes");

void launch_small_solve(int lanes, const CgArgs& a, const SmallArgs& g, hipStream_t s) {
  const dim3 grid(g.units), block(kThreads);
  switch (lanes) {
    case 8: hipLaunchKernelGGL(HIP_KERNEL_NAME(SOLVE8), grid, block, 0, s, a, g); break;
    case 16: hipLaunchKernelGGL(HIP_KERNEL_NAME(SOLVE16), grid, block, 0, s, a, g); break;
    default: hipLaunchKernelGGL(HIP_KERNEL_NAME(SOLVE32), grid, block, 0, s, a, g);
  }
}

// Workgroups of the solve that the device holds at once.
int small_resident(int lanes, int device) {
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) return 0;
  int per = 0;
  const hipError_t e =
      lanes == 8 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, SOLVE8, kThreads, 0)
      : lanes == 16 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, SOLVE16, kThreads, 0)
                    : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, SOLVE32, kThreads, 0);
  return e == hipSuccess ? per * prop.multiProcessorCount : 0;
}

int small_lanes(int32_t nslices, int32_t max_cap) {
  if (nslices < 1 || max_cap > PD_SMALL_MAX_BONDS) return 0;
  if (nslices <= PD_SMALL_UNITS / 4) return 32;
  if (nslices <= PD_SMALL_UNITS / 2) return 16;
  return nslices <= PD_SMALL_UNITS ? 8 : 0;
}

}  // namespace pd
