// Device code of the neighbour-list build, shared by prx_nl.hip
// and prx_persist.hip. See prx_nl.hip for the algorithm.
#pragma once

#include "prx_common.h"

namespace prx {

constexpr int kRangeInts = 14;  // slot range record: item_b, item_e, a0, n, then bonded ranges

constexpr int kNlThreads = 256;

__device__ __forceinline__ unsigned long long nl_below(int lane) {
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// Listed system k, by one block of kNlThreads threads.
__device__ __forceinline__ void nl_check_block(const DeviceView& v, const int32_t* ranges, int k) {
  __shared__ float sh[kNlThreads];
  const int32_t* R = ranges + k * kRangeInts;
  const int a0 = R[2], n = R[3];
  if (n <= 0) return;
  const int slot = v.slot_of[a0];
  const SlotConst& S = v.slots[slot];
  if (!S.nl || S.skin_half2 <= 0.0f) return;  // without a skin the list is built every time
  float m = 0.0f;
  auto take = [&](const float4& x, const float4& r) {
    const float dx = x.x - r.x, dy = x.y - r.y, dz = x.z - r.z;
    const float d2 = dx * dx + dy * dy + dz * dz;
    m = (d2 > m || d2 != d2) ? (d2 != d2 ? INFINITY : d2) : m;  // a non-finite position forces a build
  };
  // four atoms' loads in flight per thread: the scan is bound by load latency
  int i = threadIdx.x;
  for (; i + 3 * kNlThreads < n; i += 4 * kNlThreads) {
    float4 x[4], r[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      x[u] = v.pos[a0 + i + u * kNlThreads];
      r[u] = v.nl_xref[a0 + i + u * kNlThreads];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) take(x[u], r[u]);
  }
  for (; i < n; i += kNlThreads) take(v.pos[a0 + i], v.nl_xref[a0 + i]);
  sh[threadIdx.x] = m;
  __syncthreads();
  for (int off = kNlThreads / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) sh[threadIdx.x] = fmaxf(sh[threadIdx.x], sh[threadIdx.x + off]);
    __syncthreads();
  }
  if (threadIdx.x == 0) v.nl_flag[slot] = sh[0] > S.skin_half2 ? 1 : 0;
}

// Tile t's list, by one block: the masks of its tile pairs (I, J > I), their
// prefix counts, the row's total, the entries, and with a skin the reference
// positions of the tile's atoms. THREADS tile pairs a round: a thread each for
// the box test, the pairs in range then dealt to the waves, four loads in flight,
// and their entries written from the masks in LDS.
template <int THREADS>
__device__ __forceinline__ void nl_row_block(const DeviceView& v, int t, int force) {
  __shared__ unsigned long long masks[THREADS];
  __shared__ int prefs[THREADS];
  __shared__ int near[THREADS];
  __shared__ int totals[THREADS / 64];
  __shared__ int n_near;
  constexpr int kWaves = THREADS / 64, kBatch = 4;
  const int4 tl = v.tiles[t];
  const int slot = tl.z;
  const SlotConst& S = v.slots[slot];
  if (!S.nl || !(force || S.skin_half2 <= 0.0f || v.nl_flag[slot])) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int I = tl.w;
  const int nT = (S.n + kTile - 1) / kTile;
  const int tp0 = S.tp_base + I * (nT - 1) - (I * (I - 1)) / 2;  // record of (I, I + 1)
  const int entry0 = v.nl_row[t].y;
  const float4 li = v.tbox[2 * t], hi = v.tbox[2 * t + 1];
  if (S.skin_half2 > 0.0f && tid < tl.y) v.nl_xref[tl.x + tid] = v.pos[tl.x + tid];
  int running = 0;
  for (int J0 = I + 1; J0 < nT; J0 += THREADS) {
    const int n = min(THREADS, nT - J0), tp = tp0 + (J0 - I - 1) + tid;
    if (tid == 0) n_near = 0;
    __syncthreads();  // and the last round's entries are written
    masks[tid] = 0ull;
    bool in = false;
    if (tid < n && v.nl_tp[tp].slot >= 0) {  // else an ordinary item covers this tile pair
      const int tJ = S.tile0 + J0 + tid;
      const float4 lj = v.tbox[2 * tJ], hj = v.tbox[2 * tJ + 1];
      const float bx = fmaxf(0.0f, fmaxf(lj.x - hi.x, li.x - hj.x));
      const float by = fmaxf(0.0f, fmaxf(lj.y - hi.y, li.y - hj.y));
      const float bz = fmaxf(0.0f, fmaxf(lj.z - hi.z, li.z - hj.z));
      in = !(bx * bx + by * by + bz * bz >= S.nl_cut2);
    }
    const unsigned long long some = __ballot(in);
    int base = 0;
    if (lane == 0 && some != 0ull) base = atomicAdd(&n_near, __popcll(some));
    base = __builtin_amdgcn_readfirstlane(base);
    if (in) near[base + __popcll(some & nl_below(lane))] = tid;
    __syncthreads();
    for (int k = wave; k < n_near; k += kBatch * kWaves) {
      int e[kBatch], nJ[kBatch];
      float4 p[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        e[u] = near[min(k + u * kWaves, n_near - 1)];
        const int a = (J0 + e[u]) * kTile;
        nJ[u] = min(kTile, S.n - a);
        p[u] = v.pos[S.a0 + a + min(lane, nJ[u] - 1)];
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const float gx = fmaxf(0.0f, fmaxf(li.x - p[u].x, p[u].x - hi.x));
        const float gy = fmaxf(0.0f, fmaxf(li.y - p[u].y, p[u].y - hi.y));
        const float gz = fmaxf(0.0f, fmaxf(li.z - p[u].z, p[u].z - hi.z));
        const unsigned long long m = __ballot(lane < nJ[u] && gx * gx + gy * gy + gz * gz < S.nl_cut2);
        if (lane == 0) masks[e[u]] = m;
      }
    }
    __syncthreads();
    const unsigned long long mine = masks[tid];
    const int c = __popcll(mine);
    int incl = c;  // inclusive prefix over the lanes, in lane order
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(incl, off);
      if (lane >= off) incl += y;
    }
    if (lane == 63) totals[wave] = incl;
    __syncthreads();
    int before = running;
    for (int k = 0; k < kWaves; ++k) {
      if (k < wave) before += totals[k];
      running += totals[k];
    }
    prefs[tid] = before + incl - c;
    if (tid < n) {
      v.nl_mask[tp] = mine;
      v.nl_pref[tp] = before + incl - c;
    }
    __syncthreads();
    for (int k = wave; k < n_near; k += kWaves) {
      const int e = near[k];
      const unsigned long long m = masks[e];
      if ((m >> lane) & 1ull)
        v.nl_entries[entry0 + prefs[e] + __popcll(m & nl_below(lane))] = S.a0 + (J0 + e) * kTile + lane;
    }
    __syncthreads();
  }
  if (tid == 0) v.nl_count[t] = running;
}

}  // namespace prx
