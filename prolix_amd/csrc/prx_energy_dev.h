// Device code of the energy reduction, a launch of its own in prx_atom.hip and
// extra blocks of the chain pass in prx_pair.hip.
#pragma once

#include "prx_lanes_dev.h"
#include "prx_nl_dev.h"
#include "prolix_gb.h"

namespace prx {

// Slot range record layout (ints): item_b, item_e, a0, n, bond_b, bond_e, ang_b, ang_e,
// tors_b, tors_e, cmap_b, cmap_e, exc_b, exc_e.

// Energy reduction: one block per listed system. Each of kEnThreads threads sums
// its strided share of every term in index order, then each wave sums its 64
// lanes' terms and the waves' are added in wave order, so the result is
// deterministic. Bound by load latency and, in small systems, by the sums over
// lanes: the first element of every kind is loaded before any is added, later
// ones four iterations at a time, and the lanes are summed by exchanges in which
// a lane gives up half the terms it carries (wave_sum_terms; a butterfly per term
// through LDS took 6 of the 11 us of a 138-atom system, now 3.7 us; 64 systems of
// up to 5,000 atoms 19 us, now 12.7).
constexpr int kEnThreads = 1024;

// Elements b + t, b + t + T, ... of [b, e) (T = kEnThreads) in that order:
// acc(kind(k), energy(k)), with four elements' loads issued before their adds.
template <class K, class E, class A>
__device__ __forceinline__ void strided4(int b, int e, int t, K kind, E energy, A acc) {
  int k = b + t;
  for (; k + 3 * kEnThreads < e; k += 4 * kEnThreads) {
    int z[4];
    double x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      z[u] = kind(k + u * kEnThreads);
      x[u] = energy(k + u * kEnThreads);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) acc(z[u], x[u]);
  }
  for (; k < e; k += kEnThreads) acc(kind(k), energy(k));
}

// Sixteen terms summed over the wave: lanes 4 k to 4 k + 3 get term k.
__device__ __forceinline__ double wave_sum_terms(const double (&v)[16], int lane) {
  double h[8], g[4], f[2];
#pragma unroll
  for (int k = 0; k < 8; ++k) h[k] = add_swap<true>(v[k], v[k + 8]);
#pragma unroll
  for (int k = 0; k < 4; ++k) g[k] = add_swap<false>(h[k], h[k + 4]);
  const bool b3 = (lane & 8) != 0, b2 = (lane & 4) != 0;
#pragma unroll
  for (int k = 0; k < 2; ++k) f[k] = (b3 ? g[k + 2] : g[k]) + dpp<kDppRor8>(b3 ? g[k] : g[k + 2]);
  double e = (b2 ? f[1] : f[0]) + dpp<kDppHalfMirror>(b2 ? f[0] : f[1]);
  e += dpp<kDppXor2>(e);
  return e + dpp<kDppXor1>(e);
}

template <int THREADS>
__device__ __forceinline__ void energy_reduce_block(const DeviceView& v, const int32_t* ranges, int block, double* out) {
  constexpr int kTerms = 12, kWaves = kEnThreads / 64;
  __shared__ double part[16][kWaves];
  __shared__ double sum[16];
  const int32_t* R = ranges + block * kRangeInts;
  // the shares of kEnThreads threads, THREADS of them at a time, whatever THREADS
  // is: the same sums
  for (int t = threadIdx.x; t < kEnThreads; t += THREADS) {
    // the first element of each kind
    const auto first = [&](int b, int e, auto load) {
      if (b < e) load(min(b + t, e - 1));
    };
    double i0 = 0, i1 = 0, i2 = 0, s0 = 0, a0 = 0, xb = 0, xa = 0, xt = 0, xm = 0, xe = 0;
    int zb = 0;
    float zt = 0.0f;
    first(R[0], R[1], [&](int k) {
      i0 = v.e_items[(size_t)k * 3];
      i1 = v.e_items[(size_t)k * 3 + 1];
      i2 = v.e_items[(size_t)k * 3 + 2];
    });
    first(0, R[3], [&](int k) {
      s0 = v.e_atom[(size_t)(R[2] + k) * 2];
      a0 = v.e_atom[(size_t)(R[2] + k) * 2 + 1];
    });
    // A system's bonded ranges hold only its own entries (free entries lie
    // outside every listed range), so no entry is tested for being free; the
    // kind of a bond (bond / Urey-Bradley) and of a torsion entry (proper /
    // improper) is read beside its energy.
    first(R[4], R[5], [&](int k) { zb = v.bonds[k].idx.z; xb = v.e_bond[k]; });
    first(R[6], R[7], [&](int k) { xa = v.e_angle[k]; });
    first(R[8], R[9], [&](int k) { zt = v.tors[k].a.w; xt = v.e_tors[k]; });
    first(R[10], R[11], [&](int k) { xm = v.e_cmap[k]; });
    first(R[12], R[13], [&](int k) { xe = v.e_exc[k]; });

    const bool in_i = R[0] + t < R[1], in_a = t < R[3], in_b = R[4] + t < R[5], in_t = R[8] + t < R[9];
    double e_gbp = in_i ? i0 : 0.0, e_cl = in_i ? i1 : 0.0, e_lj = in_i ? i2 : 0.0;
    double e_self = in_a ? s0 : 0.0, e_ace = in_a ? a0 : 0.0;
    double e_bond = in_b && zb == 0 ? xb : 0.0, e_ub = in_b && zb != 0 ? xb : 0.0;
    double e_ang = R[6] + t < R[7] ? xa : 0.0;
    double e_dih = in_t && zt == 0.0f ? xt : 0.0, e_imp = in_t && zt != 0.0f ? xt : 0.0;
    double e_cm = R[10] + t < R[11] ? xm : 0.0;
    double e_ex = R[12] + t < R[13] ? xe : 0.0;

    int i = R[0] + kEnThreads + t;
    for (; i + 3 * kEnThreads < R[1]; i += 4 * kEnThreads) {
      double a[4][3];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int c = 0; c < 3; ++c) a[u][c] = v.e_items[(size_t)(i + u * kEnThreads) * 3 + c];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        e_gbp += a[u][0];
        e_cl += a[u][1];
        e_lj += a[u][2];
      }
    }
    for (; i < R[1]; i += kEnThreads) {
      e_gbp += v.e_items[(size_t)i * 3 + 0];
      e_cl += v.e_items[(size_t)i * 3 + 1];
      e_lj += v.e_items[(size_t)i * 3 + 2];
    }
    for (int k = t + kEnThreads; k < R[3]; k += kEnThreads) {
      e_self += v.e_atom[(size_t)(R[2] + k) * 2 + 0];
      e_ace += v.e_atom[(size_t)(R[2] + k) * 2 + 1];
    }
    const int t1 = t + kEnThreads;
    strided4(R[4], R[5], t1, [&](int k) { return v.bonds[k].idx.z; }, [&](int k) { return v.e_bond[k]; },
             [&](int z, double e) { if (z == 0) e_bond += e; else e_ub += e; });
    strided4(R[6], R[7], t1, [&](int) { return 0; }, [&](int k) { return v.e_angle[k]; },
             [&](int, double e) { e_ang += e; });
    strided4(R[8], R[9], t1, [&](int k) { return v.tors[k].a.w == 0.0f ? 0 : 1; }, [&](int k) { return v.e_tors[k]; },
             [&](int z, double e) { if (z == 0) e_dih += e; else e_imp += e; });
    strided4(R[10], R[11], t1, [&](int) { return 0; }, [&](int k) { return v.e_cmap[k]; },
             [&](int, double e) { e_cm += e; });
    strided4(R[12], R[13], t1, [&](int) { return 0; }, [&](int k) { return v.e_exc[k]; },
             [&](int, double e) { e_ex += e; });
    const double mine[16] = {e_bond, e_ang, e_ub, e_dih, e_imp, e_cm, e_lj, e_ex, e_gbp, e_self, e_cl, e_ace};
    const int lane = t & 63, wave = t >> 6;
    const double w = wave_sum_terms(mine, lane);
    if ((lane & 3) == 0) part[lane >> 2][wave] = w;
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < kTerms) {
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) acc += part[t][k];
    sum[t] = acc;
  }
  __syncthreads();
  if (t != 0) return;
  double terms[PRX_N_ENERGY];
  terms[PRX_E_BOND] = sum[0];
  terms[PRX_E_ANGLE] = sum[1];
  terms[PRX_E_UREY_BRADLEY] = sum[2];
  terms[PRX_E_DIHEDRAL] = sum[3];
  terms[PRX_E_IMPROPER] = sum[4];
  terms[PRX_E_CMAP] = sum[5];
  terms[PRX_E_LJ] = sum[6];
  terms[PRX_E_EXCEPTION] = sum[7];
  terms[PRX_E_GB] = sum[8] + sum[9];
  terms[PRX_E_COULOMB] = sum[10];
  terms[PRX_E_ACE] = sum[11];
  double tot = 0.0;
  for (int k = 0; k < PRX_E_TOTAL; ++k) tot += terms[k];
  terms[PRX_E_TOTAL] = tot;
  for (int k = 0; k < PRX_N_ENERGY; ++k) out[(size_t)block * PRX_N_ENERGY + k] = terms[k];
}

}  // namespace prx
