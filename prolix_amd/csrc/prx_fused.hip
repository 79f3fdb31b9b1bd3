// Fused step kernel for small systems: one workgroup per system runs K BAOAB
// steps of that system, its passes separated by workgroup barriers only.
//
// For a system of one tile a step of the graph path is six dependent launches
// of almost empty grids, so its time is launch and dependency latency (~39 us
// at 64 atoms against a few us of work), and the persistent kernel pays a
// grid-wide barrier per pass instead. Here a workgroup owns all the work of its
// system: the system's work items over its waves, its tiles' gathers side by side (one
// group of four waves per tile, each group with its own workgroup memory), its
// bonded entries over its threads. No other workgroup reads or writes that
// system's atoms, items or records, so __syncthreads (a workgroup-scope fence
// and barrier; all waves of a workgroup share one CU and its vector cache)
// orders every pass. Systems run side by side, one workgroup each, with no
// barrier between them.
//
// A tile gather holds exactly one workgroup barrier (its combine of the four
// waves' sums). In a round of gathers, a group whose tile index lies
// past the system's last tile executes one barrier in its place, so every
// wave of the workgroup meets the same number of barriers.
//
// Each pass calls the per-item and per-tile device functions of the graph's
// kernels (prx_*_dev.h) on the same items, in the same per-item and per-tile
// order, so every result is bit for bit the graph path's. Systems that take
// their pair work from a neighbour list are not run here.
#include "prx_atom_dev.h"
#include "prx_bonded_dev.h"
#include "prx_nl_dev.h"
#include "prx_pair_dev.h"

namespace prx {

namespace {

static_assert(kGW == kUnitWaves, "a group runs a unit or a tile gather");
// Threads of GROUPS groups of four waves: units and tile gathers side by side.
// One for systems of one tile, two for two tiles (registers are left to them, and several
// workgroups share a CU), else four, though they leave a wave 128 registers and spill
// some. us a step, now and with two groups for all: 64 atoms 31 and 34, 2,000 systems of
// 64 142 and 276; 100 atoms 47 and 52, 2,000 systems 377 and 418; 138 atoms 56 and 80; 500
// 198 and 259; 2,500 2,904 and 3,763.
constexpr int kTileGroups = 1, kTwoTileGroups = 2, kManyGroups = 4;
template <int GROUPS>
constexpr int kFusedThreads = GROUPS * kGW * 64;

// The bonded entries of one system (its ranges in each kind's arena).
template <int THREADS>
__device__ __forceinline__ void bonded_slot(const DeviceView& v, const int32_t* R) {
  for (int e = R[4] + (int)threadIdx.x; e < R[5]; e += THREADS) do_bond<false>(v, e);
  for (int e = R[6] + (int)threadIdx.x; e < R[7]; e += THREADS) do_angle<false>(v, e);
  for (int e = R[8] + (int)threadIdx.x; e < R[9]; e += THREADS) do_torsion<false>(v, e);
  for (int e = R[10] + (int)threadIdx.x; e < R[11]; e += THREADS) do_cmap<false>(v, e);
  for (int e = R[12] + (int)threadIdx.x; e < R[13]; e += THREADS) do_exception<false>(v, e);
}

// One round of tile gathers: group g of four waves gathers tile t + g, or,
// past the last tile, takes the one barrier that gather would have held.
// Then the round's barrier, before the workgroup memory is used again.
template <class F>
__device__ __forceinline__ void gather_round(int t, int t1, int grp, F&& gather) {
  if (t + grp < t1)
    gather(t + grp);
  else
    __syncthreads();
  __syncthreads();
}

// One pair pass of a system, items i0 to i1 - 1. A system of one tile: its item on
// four waves. Others: up to kFusedPairs items on two waves each, more on one, without
// barriers in between. us a step with an item on four, two and one wave: 192 atoms (6
// items) 76, 61, -; 256 (10) 104, 100, 88; 500 (36) 285, 247, 198.
constexpr int kFusedPairs = 8;

template <class Pass, int GROUPS>
__device__ __forceinline__ void pair_pass(const DeviceView& v, int i0, int i1, int wave, int grp, int uw, float4* L) {
  if constexpr (GROUPS == kTileGroups) {
    pair_unit<Pass, kUnitWaves, false, true>(v, PairUnit{i0, 1, kUnitWaves}, uw, true, L);
    __syncthreads();
  } else {
    const bool pairs = i1 - i0 <= kFusedPairs;
    const int step = GROUPS * (pairs ? 2 : kUnitWaves);
    for (int k = i0 + (pairs ? 0 : wave); k < i1; k += step) {
      const int first = pairs ? k + 2 * grp : k;
      if (first >= i1) {  // the barriers that the unit would have held
        __syncthreads();
        __syncthreads();
      } else {
        const PairUnit u = {first, (int16_t)(pairs ? min(2, i1 - first) : 1), (int16_t)(pairs ? 2 : 1)};
        pair_unit<Pass, 2 * kUnitWaves, true>(v, u, pairs ? uw : 0, pairs, pairs ? L : L + uw * kAnyWaveLds);
      }
      if (pairs) __syncthreads();
    }
    if (!pairs) __syncthreads();
  }
}

// Block b: the b-th listed system, ranges row b (item_b, item_e, a0, n, then
// the bonded ranges).
template <int GROUPS>
__global__ __launch_bounds__(kFusedThreads<GROUPS>) void k_fused_steps(DeviceView v, const int32_t* ranges, int n_steps) {
  __shared__ float4 ulds[GROUPS][GROUPS == kTileGroups ? kAnyGroupLds : kUnitWaves * kAnyWaveLds];
  __shared__ GatherLds glds[GROUPS];
  const int32_t* R = ranges + (size_t)blockIdx.x * kRangeInts;
  const int a0 = R[2], n = R[3];
  if (n <= 0) return;
  const SlotConst& S = v.slots[v.slot_of[a0]];
  const int t0 = S.tile0;
  const int t1 = t0 + (n + kTile - 1) / kTile;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int grp = wave / kGW;
  const int uw = unit_wave();
  float4* const L = ulds[grp];
  GatherLds& G = glds[grp];

  // B A O A of the first step from the stored force, then the tile boxes
  for (int g = a0 + (int)threadIdx.x; g < a0 + n; g += kFusedThreads<GROUPS>) step_begin_atom(v, g);
  __syncthreads();
  for (int t = t0 + wave; t < t1; t += GROUPS * kGW) tile_box_wave(v, t);
  __syncthreads();

  for (int k = 0; k < n_steps; ++k) {
    bonded_slot<kFusedThreads<GROUPS>>(v, R);
    pair_pass<BornPass, GROUPS>(v, R[0], R[1], wave, grp, uw, L);
    for (int t = t0; t < t1; t += GROUPS)
      gather_round(t, t1, grp, [&](int tt) { born_gather_tile(v, tt, G); });
    pair_pass<ForcePass<false>, GROUPS>(v, R[0], R[1], wave, grp, uw, L);
    for (int t = t0; t < t1; t += GROUPS)
      gather_round(t, t1, grp, [&](int tt) { force_gather_tile<false>(v, tt, G); });
    pair_pass<ChainPass, GROUPS>(v, R[0], R[1], wave, grp, uw, L);
    const int mode = k + 1 == n_steps ? 2 : 1;  // the last step stops after B(F)
    for (int t = t0; t < t1; t += GROUPS)
      gather_round(t, t1, grp, [&](int tt) { chain_gather_tile(v, tt, mode, G); });
  }
}

}  // namespace

void launch_fused_steps(const DeviceView& v, const int32_t* slot_ranges, int n_slots, int max_atoms, int n_steps,
                        hipStream_t s) {
  // every tile gather must reach its barrier: no stopped-system early return here
  DeviceView fv = v;
  fv.skip_done = 0;
  if (n_slots <= 0 || n_steps <= 0) return;
  const auto launch = [&](auto groups) {
    constexpr int G = decltype(groups)::value;
    hipLaunchKernelGGL(k_fused_steps<G>, dim3(n_slots), dim3(kFusedThreads<G>), 0, s, fv, slot_ranges, n_steps);
  };
  if (max_atoms <= kTile)
    launch(std::integral_constant<int, kTileGroups>());
  else if (max_atoms <= 2 * kTile)
    launch(std::integral_constant<int, kTwoTileGroups>());
  else
    launch(std::integral_constant<int, kManyGroups>());
}

}  // namespace prx
