// All-pairs passes of the GB-OBC2 energy/force evaluation on gfx950.
//
// A work item is a 64x64 tile pair I <= J of one system, evaluated in 8x8
// patches of 8x8 pairs (prx_pair_dev.h): the wave's columns and their sums
// stay in registers, rows come from LDS. A wave stores the row and column
// sums of its item in the item's own slots of the partial buffer (plain
// stores, no atomics); the tile gathers of prx_atom.hip add them up in a fixed
// order, so results are bitwise reproducible.
//
// Pass 1 (Born sums, generalized_born.py:211-263 with :32-94):
//     I_i += I(r; rho_i, sr_j),  I_j += I(r; rho_j, sr_i)
// Pass 2 (GB + Coulomb + LJ forces and dE/dB, generalized_born.py:97-208,
//     optimization.py:21-297): GB over every pair, Coulomb/LJ with exclusion
//     scales and the optional cutoff.
// Pass 3 (Born chain rule, generalized_born.py:651-706):
//     F -= (c_i dI_ij/dr + c_j dI_ji/dr) dr/dx, c = dE/dB * dB/dI.
//
// Diagonal tiles (I == J) visit each unordered pair once: the patches above
// the diagonal, and the pairs p > q of those on it.
//
// Systems with a cutoff: the Born pass classifies each item from its two
// tiles' bounding boxes (near / straddle / far, stored for the later passes
// and the gathers). Far items skip LJ and Coulomb, and with the neighbour-list
// GB form (generalized_born.py:266-415, gb_cut) skip every pass; straddling
// items test r^2 < cutoff^2 per pair.
#include <type_traits>

#include "prx_bonded_dev.h"
#include "prx_energy_dev.h"
#include "prx_pair_dev.h"

namespace prx {

// Blocks of the pair kernels: one, two or four waves that take an item each, or
// four waves that take a unit of the list (items of systems that differ in waves
// per item).
enum { kWaveBlocks = 1, kPairBlocks = 2, kQuadBlocks = 4, kUnitBlocks = 0 };
template <int BLOCKS>
constexpr int kThreads = 64 * (BLOCKS == kUnitBlocks ? kUnitWaves : BLOCKS);

template <int BLOCKS, class Pass>
__device__ __forceinline__ void pair_block(const DeviceView& v, int b, int nb) {
  const int i = unit_id(v, b, nb);
  if constexpr (BLOCKS == kWaveBlocks) {
    __shared__ float4 mem[kWaveLds<Pass>];
    pair_wave<Pass>(v, i, mem);
  } else if constexpr (BLOCKS == kPairBlocks) {
    __shared__ float4 mem[2 * kWaveLds<Pass>];
    pair_unit<Pass, 2, false>(v, PairUnit{i, 1, 2}, unit_wave<2>(), true, mem);
  } else if constexpr (BLOCKS == kQuadBlocks) {
    __shared__ float4 mem[Pass::Quarter::kSize];
    pair_unit<Pass, kUnitWaves, false, true>(v, PairUnit{i, 1, kUnitWaves}, unit_wave(), true, mem);
  } else {
    __shared__ float4 mem[kGroupLds<Pass>];
    const PairUnit u = v.units[i];
    pair_unit<Pass, kUnitWaves, false>(v, u, unit_wave(), u.shares > 1, mem);
  }
}

template <int BLOCKS>
__global__ __launch_bounds__(kThreads<BLOCKS>) PRX_OCCUPANCY void k_born_pairs(DeviceView v) {
  pair_block<BLOCKS, BornPass>(v, blockIdx.x, gridDim.x);
}

template <int BLOCKS, bool ENERGY>
__global__ __launch_bounds__(kThreads<BLOCKS>) PRX_FORCE_OCCUPANCY(BLOCKS, ENERGY) void k_force_pairs(DeviceView v) {
  pair_block<BLOCKS, ForcePass<ENERGY>>(v, blockIdx.x, gridDim.x);
}

template <int BLOCKS>
__global__ __launch_bounds__(kThreads<BLOCKS>) PRX_OCCUPANCY void k_chain_pairs(DeviceView v) {
  pair_block<BLOCKS, ChainPass>(v, blockIdx.x, gridDim.x);
}

// The chain pass with the energy reduction in the same launch: blocks below
// n_slots take a system's energies each, which are complete before the pass, the
// rest the pass's items or units.
template <int BLOCKS>
__global__ __launch_bounds__(kThreads<BLOCKS>) void k_chain_pairs_energies(DeviceView v, const int32_t* ranges,
                                                                           int n_slots, double* out) {
  const int b = (int)blockIdx.x;
  if (b < n_slots)
    energy_reduce_block<kThreads<BLOCKS>>(v, ranges, b, out);
  else
    pair_block<BLOCKS, ChainPass>(v, b - n_slots, (int)gridDim.x - n_slots);
}

// The Born pass with the bonded terms in the same launch: blocks below
// n_pair are the pair kernel's (its XCD-aware order over those blocks), the
// rest take one bonded entry per thread. Both read positions only and the
// bonded records are read by the chain gather, so the merged launch saves the
// bonded kernel's graph node where that kernel would run in line; results are
// bit for bit those of the two kernels.
template <int BLOCKS, bool ENERGY>
__global__ __launch_bounds__(kThreads<BLOCKS>) PRX_OCCUPANCY void k_born_pairs_bonded(DeviceView v, int n_pair) {
  const int b = (int)blockIdx.x;
  if (b < n_pair) {
    pair_block<BLOCKS, BornPass>(v, b, n_pair);
    return;
  }
  const int e = (b - n_pair) * kThreads<BLOCKS> + (int)threadIdx.x;
  if (e < bonded_entries(v)) bonded_entry<ENERGY>(v, e);
}

// Blocks of a list: one, two or four waves per item where every item takes as many,
// else units.
// Two-wave blocks free their slots as soon as one item is done, and read no unit list:
// 8,000 atoms 144 us an evaluation, 148 with units of two items.
static inline int list_blocks(const DeviceView& v) { return v.shares; }
static inline int pair_blocks(const DeviceView& v, int blocks) { return blocks == kUnitBlocks ? v.n_units : v.n_items; }

// launch(std::integral_constant<int, BLOCKS>) with the list's blocks.
template <class F>
static void by_blocks(const DeviceView& v, F&& launch) {
  static_assert(kQuadBlocks == kUnitWaves, "shares name the blocks");
  switch (list_blocks(v)) {
    case kWaveBlocks: return launch(std::integral_constant<int, kWaveBlocks>());
    case kPairBlocks: return launch(std::integral_constant<int, kPairBlocks>());
    case kQuadBlocks: return launch(std::integral_constant<int, kQuadBlocks>());
    default: return launch(std::integral_constant<int, kUnitBlocks>());
  }
}

template <bool ENERGY>
static void born_pairs_bonded(const DeviceView& v, hipStream_t s) {
  by_blocks(v, [&](auto b) {
    constexpr int B = decltype(b)::value, nt = kThreads<B>;
    const int np = pair_blocks(v, B), nb = np + (bonded_entries(v) + nt - 1) / nt;
    if (nb > 0) hipLaunchKernelGGL((k_born_pairs_bonded<B, ENERGY>), dim3(nb), dim3(nt), 0, s, v, np);
  });
}

void launch_born_pairs_bonded(const DeviceView& v, bool energy, hipStream_t s) {
  if (energy)
    born_pairs_bonded<true>(v, s);
  else
    born_pairs_bonded<false>(v, s);
}

void launch_born_pairs(const DeviceView& v, hipStream_t s) {
  if (v.n_items == 0) return;
  by_blocks(v, [&](auto b) {
    constexpr int B = decltype(b)::value;
    hipLaunchKernelGGL(k_born_pairs<B>, dim3(pair_blocks(v, B)), dim3(kThreads<B>), 0, s, v);
  });
}

template <bool ENERGY>
static void force_pairs(const DeviceView& v, hipStream_t s) {
  by_blocks(v, [&](auto b) {
    constexpr int B = decltype(b)::value;
    hipLaunchKernelGGL((k_force_pairs<B, ENERGY>), dim3(pair_blocks(v, B)), dim3(kThreads<B>), 0, s, v);
  });
}

void launch_force_pairs(const DeviceView& v, bool energy, hipStream_t s) {
  if (v.n_items == 0) return;
  if (energy)
    force_pairs<true>(v, s);
  else
    force_pairs<false>(v, s);
}

void launch_chain_pairs(const DeviceView& v, hipStream_t s) {
  if (v.n_items == 0) return;
  by_blocks(v, [&](auto b) {
    constexpr int B = decltype(b)::value;
    hipLaunchKernelGGL(k_chain_pairs<B>, dim3(pair_blocks(v, B)), dim3(kThreads<B>), 0, s, v);
  });
}

// In lists of four-wave units the reduction hides behind the pass (138 atoms 68.3 us
// an evaluation with a launch of its own, 66.0 in this one, 1,237 atoms 75.7 and
// 71.5), also that of a large system which a smaller one brings into such a list
// (energies add 10 us to the forces of 130 + 8,300 atoms, 17 to those of 130 + 12,000). The
// other lists' blocks of 64 or 128 threads would take two or four times as long
// over a system.
bool launch_chain_pairs_energies(const DeviceView& v, const int32_t* ranges, int n_slots, double* out, hipStream_t s) {
  if (v.n_items == 0) return false;
  const int blocks = list_blocks(v);
  if (blocks == kQuadBlocks)
    hipLaunchKernelGGL(k_chain_pairs_energies<kQuadBlocks>, dim3(n_slots + v.n_items), dim3(kThreads<kQuadBlocks>), 0, s,
                       v, ranges, n_slots, out);
  else if (blocks == kUnitBlocks)
    hipLaunchKernelGGL(k_chain_pairs_energies<kUnitBlocks>, dim3(n_slots + v.n_units), dim3(kThreads<kUnitBlocks>), 0, s,
                       v, ranges, n_slots, out);
  else
    return false;
  return true;
}

}  // namespace prx
