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
//   * each lane keeps the 3x3 blocks of its slots in registers for the whole
//     solve (at most 15 blocks, 180 VGPRs): a product gathers 48 bytes per
//     bond and multiplies;
//   * the workgroups exchange z, p and the partial sums through global
//     memory without leaving the kernel.
// Measured at 8,000 rows, 11 iterations: assembly 93 -> 31 us, solve about
// 590 (44 launches) -> 247 us, the step 744 -> 315 us; at 288 rows the step
// 400 -> 147 us.
#include <math.h>

#include "pd_bond.h"

namespace pd {

namespace {

constexpr int kThreads = PD_SMALL_THREADS;

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
#pragma unroll
  for (int m = R / 2; m >= 1; m >>= 1) v = v + __shfl_xor(v, m, 64);
  return v;
}

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

__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Fold of one partial row over tiles [t0, t0 + nt), nt <= 64, by one wave:
// fold_partials' tree.  Lane t joins the units of tile t's four slices
// (levels 2^(K-1) .. 1 of the butterfly within a slice, then (w0 + w1) +
// (w2 + w3)); tiles beyond nt add 0.0.  WAIT: the partials are written by
// running workgroups, each is awaited until it is set or `until` (100 MHz
// clock) has passed; then *late is raised.
template <int K, bool WAIT>
__device__ __forceinline__ double fold_units(const double* part, int t0, int nt, int nslices,
                                             int lane, unsigned long long until, bool* late) {
  constexpr int U = 1 << K;
  double w[4][U];
  const bool mine = lane < nt;
  bool ready = false;
  for (unsigned spin = 0; !ready; ++spin) {
    ready = true;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = (t0 + lane) * 4 + j;
      const bool in = mine && s < nslices;
#pragma unroll
      for (int c = 0; c < U; ++c) {
        w[j][c] = in ? get(part + (s << K) + c) : 0.0;
        if (WAIT && is_unset(w[j][c])) ready = false;
      }
    }
    if (!WAIT) break;
    ready = __all(ready);
    if (!ready && (spin & 15) == 15 && wall_clock64() > until) {
      *late = true;
      break;
    }
  }
  double ws[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (K == 0) ws[j] = w[j][0];
    if constexpr (K == 1) ws[j] = w[j][0] + w[j][1];
    if constexpr (K == 2) ws[j] = (w[j][0] + w[j][2]) + (w[j][1] + w[j][3]);
  }
  double acc = 0.0;
  if (mine) acc = acc + ((ws[0] + ws[1]) + (ws[2] + ws[3]));
  const double v = wave_sum(acc);
  return (v + 0.0) + (0.0 + 0.0);
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
// 2 L additions in a row.
// ---------------------------------------------------------------------------
template <int L, bool SHARED>
__device__ __forceinline__ void small_assemble(const AsmArgs& a, const SmallArgs& g,
                                               double* lds) {
  constexpr int R = Unit<L>::R, K = Unit<L>::K;
  constexpr int CH = 2 * L, CP = CH + 1;  // slots per chunk and its padded stride
  constexpr int ROW = 13 * CP;            // LDS doubles per row
  constexpr int ROLES = 15;               // 13 sums, the smallest and the largest stretch
  constexpr int NR = (ROLES + L - 1) / L;
  const int unit = xcd_tile(blockIdx.x, gridDim.x);
  const int s = unit >> K;
  const int i = threadIdx.x / L, j = threadIdx.x % L;  // row of the unit, lane of the row
  const int pl = (i << K) + (unit & ((1 << K) - 1));
  const int p = s * 64 + pl;
  const bool vis = p < a.n && a.act[p] != PD_INVISIBLE;
  double* tr = lds + i * ROW;
  const int64_t base = a.slice_off[s];
  int top = vis ? a.top[p] : -1;
  const int otop = top;
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
  bool zero_len = false;
  double acc[NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) acc[k] = j + k * L == 14 ? -INFINITY : 0.0;

  // geometry, stretch and breaking test of slot k (k <= top)
  struct Bond {
    double4 u;
    double d0, e0, e1, e2, dij, yd, dr;
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
    bond_dir<SHARED>(pos_p, xq, b.e0, b.e1, b.e2, b.dij);
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
        if (in && SHARED) zero_len = zero_len || b[u].dij == 0.0;
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
          if (SHARED) zero_len = zero_len || t.dij == 0.0;
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
      bond_jac_sc<SHARED>(t.e0, t.e1, t.e2, t.dij, t.d0, sc, F00, F01, F02, F11, F12, F22);
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
    }
    wave_fence();
    const int m = min(CH, top + 1 - c0);
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int role = j + k * L;
      if (role < ROLES) {
        const double* t = tr + min(role, 12) * CP;
        double v = acc[k];
        int e = 0;
        if (role < 13) {
          for (; e + 8 <= m; e += 8) {
            double x[8];
#pragma unroll
            for (int w = 0; w < 8; ++w) x[w] = t[e + w];
#pragma unroll
            for (int w = 0; w < 8; ++w) v += x[w];
          }
          for (; e < m; ++e) v += t[e];
        } else if (role == 13) {
          for (; e < m; ++e) v = t[e] < v ? t[e] : v;
        } else {
          for (; e < m; ++e) v = t[e] > v ? t[e] : v;
        }
        acc[k] = v;
      }
    }
    wave_fence();
  }
  // the row's sums to the unit's owner lanes (the first R threads)
  __syncthreads();
  double* sum = lds;  // [R][16]
#pragma unroll
  for (int k = 0; k < NR; ++k)
    if (j + k * L < ROLES) sum[i * 16 + j + k * L] = acc[k];
  int* tops = (int*)(lds + R * 16);  // [R]
  if (j == 0) tops[i] = top;
  const bool zany = __any(zero_len);
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
  (void)otop;
  const double v0 = unit_sum<R>(t_rz), v1 = unit_sum<R>(t_rr), v2 = unit_sum<R>(t_bb);
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    broken += __shfl_xor(broken, m, 64);
    live += __shfl_xor(live, m, 64);
  }
  if (threadIdx.x == 0) {
    g.start[unit] = v0;
    g.start[g.units + unit] = v1;
    g.start[2 * g.units + unit] = v2;
#pragma unroll
    for (int k = 0; k < 6; ++k) g.part[k * g.units + unit] = unset();
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
// The CG solve of a step in one launch, every workgroup resident: CUSP's loop as the general kernels run it (k_cg_spmv,
// k_cg_update, k_cg_beta, k_cg_dir), the same sums in the same order.
//
// An iteration: every lane gathers z and the previous direction of its
// slots' neighbours, forms p = z + beta p, multiplies its blocks and leaves
// the terms in LDS; lanes 0..2 of a row add them in list order on top of
// the diagonal term.  The first R threads then own a row each: <y, p>, and
// once every unit's partial is there alpha, x, r, z; once <r, z> and <r, r>
// are there, beta and the monitor test.  A unit's partial doubles as its
// arrival: partials are awaited until they are set, and those of the
// phase before are unset again once the next phase's are complete (all
// units have read them by then).  z and p go through global memory with an
// agent release ahead of the partial and an agent acquire after the wait,
// by one wave per workgroup (by all eight, the cache maintenance alone took
// 30 to 60 us per round; by one it is not seen).
//
// Every wait ends: after g.spin_ticks of the 100 MHz clock a workgroup
// raises *g.aborted and leaves.  The position update behind it then does
// nothing, and the host puts the start values back (the assembly record
// holds them) and solves with the general kernels.
// ---------------------------------------------------------------------------
template <int L, int M, int MC>
__global__ __launch_bounds__(kThreads) void k_small_solve(CgArgs a, SmallArgs g) {
  constexpr int R = Unit<L>::R, K = Unit<L>::K;
  constexpr int CH = MC * L, CP = CH + 3;  // slots per chunk, padded stride
  __shared__ double T[R * 3 * CP];         // terms
  __shared__ double Y[R * 3];
  __shared__ double Mi[6 * R];  // the rows' inverse blocks
  __shared__ double ctl[2];     // beta, and whether the loop goes on
  const int units = g.units;
  const int unit = xcd_tile(blockIdx.x, gridDim.x);
  const int s = unit >> K, cl = unit & ((1 << K) - 1);
  const int i = threadIdx.x / L, j = threadIdx.x % L;
  const int pl = (i << K) + cl;
  const int p = s * 64 + pl;
  const bool row = p < a.A.n;
  const int top = row ? a.A.top[p] : -1;
  const unsigned long long until = wall_clock64() + g.spin_ticks;
  const int spec = spec_of(a.batch, s >> 2);
  int t0, nt;
  spec_range_of(a.batch, spec, (a.A.n + PD_BLOCK - 1) / PD_BLOCK, t0, nt);
  if (unit == 0 && threadIdx.x == 0) *g.h_cnt = *g.counters;
  // a tile between specimens: its rows are invisible, nobody awaits its sums
  if ((s >> 2) >= t0 + nt) return;
  // the slots' blocks (zero past the list's end, where nothing adds them)
  int q[M];
  double B[M][6];
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
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int k = m * L + j;
#pragma unroll
      for (int c = 0; c < 6; ++c) B[m][c] = 0.0;
      if (q[m] >= 0) {
        const double l0 = ntl(lp + (int64_t)k * 64);
        const double4 xq = a.A.pos[q[m]];
        double e0, e1, e2, dij, F00, F01, F02, F11, F12, F22;
        if (shared) {
          bond_dir<true, true>(pos_p, xq, e0, e1, e2, dij);
          bond_jac<true>(e0, e1, e2, dij, l0, cb, F00, F01, F02, F11, F12, F22);
        } else {
          bond_dir(pos_p, xq, e0, e1, e2, dij);
          bond_jac(e0, e1, e2, dij, l0, cb, F00, F01, F02, F11, F12, F22);
        }
        B[m][0] = (F00 * -1.0) * dt2;
        B[m][1] = (F01 * -1.0) * dt2;
        B[m][2] = (F02 * -1.0) * dt2;
        B[m][3] = (F11 * -1.0) * dt2;
        B[m][4] = (F12 * -1.0) * dt2;
        B[m][5] = (F22 * -1.0) * dt2;
        if (a.vals)
          store_block(a.vals, base + k, pl, B[m][0], B[m][1], B[m][2], B[m][3], B[m][4],
                      B[m][5]);
      } else {
        q[m] = pc;  // a gather in bounds, its term unused
      }
    }
  }
  // lanes 0..2 of a row: row j of the diagonal block
  double g0 = 0.0, g1 = 0.0, g2 = 0.0;
  if (j < 3) {
    const double* dg = a.A.diag + (int64_t)s * 384 + pl;
    g0 = dg[j == 0 ? 0 : j == 1 ? 64 : 128];
    g1 = dg[j == 0 ? 64 : j == 1 ? 192 : 256];
    g2 = dg[j == 0 ? 128 : j == 1 ? 256 : 320];
  }
  // the first R threads own a row each
  const int ol = (threadIdx.x << K) + cl;
  const int op = s * 64 + ol;
  const bool own = threadIdx.x < R && op < a.A.n;
  double x0 = 0.0, x1 = 0.0, x2 = 0.0, r0 = 0.0, r1 = 0.0, r2 = 0.0;
  double z0 = 0.0, z1 = 0.0, z2 = 0.0, p0 = 0.0, p1 = 0.0, p2 = 0.0;
  bool fr = false;
  if (own) {
    const double4 xx = a.x[op], rr = a.r[op];
    x0 = xx.x;
    x1 = xx.y;
    x2 = xx.z;
    r0 = rr.x;
    r1 = rr.y;
    r2 = rr.z;
    const double* e = g.ex + 6 * (int64_t)op;
    z0 = e[0];
    z1 = e[1];
    z2 = e[2];
    fr = a.bc[op] == 0;
    if (a.precond) {
      const double* m = a.minv + (int64_t)s * 384 + ol;
#pragma unroll
      for (int c = 0; c < 6; ++c) Mi[c * R + threadIdx.x] = m[c * 64];
    }
  }
  const int lane = threadIdx.x & 63;
  const bool lead = threadIdx.x < 64;  // the wave of the owners
  bool late = false;
  double rz = 0.0, rr = 0.0, tol = 0.0, bnorm = 0.0, rnorm = 0.0, alpha = 0.0, beta = 0.0,
         yp = 0.0;
  int iter = 0;
  bool done = false, conv = false;
  if (lead) {
    rz = fold_units<K, false>(g.start, t0, nt, g.nslices, lane, 0, &late);
    rr = fold_units<K, false>(g.start + units, t0, nt, g.nslices, lane, 0, &late);
    const double bb = fold_units<K, false>(g.start + 2 * units, t0, nt, g.nslices, lane, 0, &late);
    bnorm = sqrt(bb);
    tol = g.rtol * bnorm;
    rnorm = sqrt(rr);
    if (rnorm <= tol) {
      done = true;
      conv = true;
    } else if (g.max_iter <= 0) {
      done = true;
    }
    if (threadIdx.x == 0) {
      ctl[0] = 0.0;
      ctl[1] = done ? 0.0 : 1.0;
    }
  }
  __syncthreads();
  const int64_t exn = 6 * (int64_t)a.A.n;
  double* P_yp = g.part;
  double* P_rz = g.part + 2 * units;
  double* P_rr = g.part + 4 * units;
  for (int it = 0; ctl[1] != 0.0; ++it) {
    const double bt = ctl[0];
    const double* ex = g.ex + (it & 1 ? exn : 0);
    double acc = 0.0;
    if (j < 3 && row) {
      const double* e = ex + 6 * (int64_t)p;
      double v0 = e[0], v1 = e[1], v2 = e[2];
      if (it > 0) {
        v0 = v0 + bt * e[3];
        v1 = v1 + bt * e[4];
        v2 = v2 + bt * e[5];
      }
      acc = g0 * v0 + g1 * v1 + g2 * v2;
    }
#pragma unroll
    for (int m0 = 0; m0 < M; m0 += MC) {
#pragma unroll
      for (int m = m0; m < m0 + MC; ++m) {
        if (m >= M) break;
        const dbl2v* e = (const dbl2v*)(ex + 6 * (int64_t)q[m]);
        const dbl2v ea = e[0], eb = e[1], ec = e[2];
        double v0 = ea.x, v1 = ea.y, v2 = eb.x;
        if (it > 0) {
          v0 = v0 + bt * eb.y;
          v1 = v1 + bt * ec.x;
          v2 = v2 + bt * ec.y;
        }
        double u0, u1, u2;
        blk6(B[m][0], B[m][1], B[m][2], B[m][3], B[m][4], B[m][5],
             make_double4(v0, v1, v2, 0.0), u0, u1, u2);
        double* o = T + i * 3 * CP + (m - m0) * L + j;
        o[0] = u0;
        o[CP] = u1;
        o[2 * CP] = u2;
      }
      wave_fence();
      if (j < 3) {
        const double* t = T + (i * 3 + j) * CP;
        const int cnt = min(CH, top + 1 - m0 * L);
        int e = 0;
        for (; e + 8 <= cnt; e += 8) {
          double h[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) h[u] = t[e + u];
#pragma unroll
          for (int u = 0; u < 8; ++u) acc += h[u];
        }
        for (; e < cnt; ++e) acc += t[e];
      }
      wave_fence();
    }
    if (j < 3) Y[i * 3 + j] = acc;
    __syncthreads();
    if (lead) {
      const int b = it & 1;
      double t_yp = 0.0, y0 = 0.0, y1 = 0.0, y2 = 0.0;
      if (own) {
        y0 = Y[threadIdx.x * 3];
        y1 = Y[threadIdx.x * 3 + 1];
        y2 = Y[threadIdx.x * 3 + 2];
        if (it > 0) {
          p0 = z0 + bt * p0;
          p1 = z1 + bt * p1;
          p2 = z2 + bt * p2;
        } else {
          p0 = z0;
          p1 = z1;
          p2 = z2;
        }
        t_yp = (y0 * p0 + y1 * p1) + y2 * p2;
      }
      const double vy = unit_sum<R>(t_yp);
      if (lane == 0) put(P_yp + b * units + unit, vy);
      if (own) {  // the direction the next iteration gathers
        double* e = g.ex + (b ? 0 : exn) + 6 * (int64_t)op;
        e[3] = p0;
        e[4] = p1;
        e[5] = p2;
      }
      yp = fold_units<K, true>(P_yp + b * units, t0, nt, g.nslices, lane, until, &late);
      alpha = rz / yp;
      double t_rz = 0.0, t_rr = 0.0;
      if (own) {
        x0 = alpha * p0 + x0;
        x1 = alpha * p1 + x1;
        x2 = alpha * p2 + x2;
        if (fr) {
          const double na = -alpha;
          r0 = na * y0 + r0;
          r1 = na * y1 + r1;
          r2 = na * y2 + r2;
        }
        z0 = r0;
        z1 = r1;
        z2 = r2;
        if (a.precond) {
          const double* m = Mi + threadIdx.x;
          const double m00 = m[0], m01 = m[R], m02 = m[2 * R], m11 = m[3 * R], m12 = m[4 * R],
                       m22 = m[5 * R];
          z0 = m00 * r0 + m01 * r1 + m02 * r2;
          z1 = m01 * r0 + m11 * r1 + m12 * r2;
          z2 = m02 * r0 + m12 * r1 + m22 * r2;
        }
        double* e = g.ex + (b ? 0 : exn) + 6 * (int64_t)op;
        e[0] = z0;
        e[1] = z1;
        e[2] = z2;
        t_rz = (r0 * z0 + r1 * z1) + r2 * z2;
        t_rr = (r0 * r0 + r1 * r1) + r2 * r2;
      }
      const double vz = unit_sum<R>(t_rz), vr = unit_sum<R>(t_rr);
      if (lane == 0 && it > 0) {  // all units have read the previous <r, z>
        put(P_rz + (b ^ 1) * units + unit, unset());
        put(P_rr + (b ^ 1) * units + unit, unset());
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      if (lane == 0) {
        put(P_rz + b * units + unit, vz);
        put(P_rr + b * units + unit, vr);
      }
      const double nrz =
          fold_units<K, true>(P_rz + b * units, t0, nt, g.nslices, lane, until, &late);
      rr = fold_units<K, true>(P_rr + b * units, t0, nt, g.nslices, lane, until, &late);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      // all units have read this iteration's <y, p>
      if (lane == 0) put(P_yp + b * units + unit, unset());
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

// blocks per lane (L * M >= PD_SMALL_MAX_BONDS) and slots per chunk
#define SOLVE8 k_small_solve<8, 15, 3>
#define SOLVE16 k_small_solve<16, 8, 8>
#define SOLVE32 k_small_solve<32, 4, 4>
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
