// Per-atom kernels: Born-radius finish, chain-rule factors, BAOAB halves,
// Philox noise, copies and deterministic per-system reductions.
#include "prx_atom_dev.h"
#include "prx_energy_dev.h"

namespace prx {
// One block per tile: the gathers and finishes of prx_atom_dev.h.
__global__ __launch_bounds__(256) void k_born_gather(DeviceView v, float* out) {
  __shared__ GatherLds G;
  if ((int)blockIdx.x >= v.n_tiles) return;
  born_gather_tile(v, blockIdx.x, G, out);
}

template <bool ENERGY>
__global__ __launch_bounds__(256) void k_force_gather(DeviceView v) {
  __shared__ GatherLds G;
  if ((int)blockIdx.x >= v.n_tiles) return;
  force_gather_tile<ENERGY>(v, blockIdx.x, G);
}

__global__ __launch_bounds__(256) void k_chain_gather(DeviceView v, int mode, float* out) {
  __shared__ GatherLds G;
  if ((int)blockIdx.x >= v.n_tiles) return;
  chain_gather_tile(v, blockIdx.x, mode, G, out);
}

__global__ void k_step_begin(DeviceView v) { step_begin_atom(v, blockIdx.x * blockDim.x + threadIdx.x); }

// ---------------------------------------------------------------------------
// Block reductions (fixed tree: deterministic)
// ---------------------------------------------------------------------------
constexpr int kRedThreads = 256;

__device__ double block_sum(double x, double* sh) {
  const int t = threadIdx.x;
  sh[t] = x;
  __syncthreads();
  for (int off = kRedThreads / 2; off > 0; off >>= 1) {
    if (t < off) sh[t] += sh[t + off];
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(kEnThreads) void k_energy_reduce(DeviceView v, const int32_t* ranges, double* out) {
  energy_reduce_block<kEnThreads>(v, ranges, blockIdx.x, out);
}

__global__ __launch_bounds__(kRedThreads) void k_kinetic(DeviceView v, const int32_t* ranges,
                                                         double* out) {
  __shared__ double sh[kRedThreads];
  const int32_t* R = ranges + blockIdx.x * kRangeInts;
  double ke = 0.0;
  for (int i = threadIdx.x; i < R[3]; i += kRedThreads) {
    const float4 p = v.mom[R[2] + i];
    ke += 0.5 * ((double)p.x * p.x + (double)p.y * p.y + (double)p.z * p.z) * (double)p.w;
  }
  ke = block_sum(ke, sh);
  if (threadIdx.x == 0) out[blockIdx.x] = ke;
}

// Positions minus the system's mass-weighted centre of mass (masses from the
// stored 1/m in mom.w), FP64 sums; one block per listed system.
__global__ __launch_bounds__(kRedThreads) void k_recenter_com(DeviceView v, const int32_t* ranges) {
  __shared__ double sh[kRedThreads];
  const int32_t* R = ranges + blockIdx.x * kRangeInts;
  double sm = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
  for (int i = threadIdx.x; i < R[3]; i += kRedThreads) {
    const int g = R[2] + i;
    const double m = 1.0 / (double)v.mom[g].w;
    const float4 x = v.pos[g];
    sm += m; sx += m * x.x; sy += m * x.y; sz += m * x.z;
  }
  const double mt = block_sum(sm, sh) + 1e-30;
  const double cx = block_sum(sx, sh) / mt, cy = block_sum(sy, sh) / mt, cz = block_sum(sz, sh) / mt;
  for (int i = threadIdx.x; i < R[3]; i += kRedThreads) {
    const int g = R[2] + i;
    float4 x = v.pos[g];
    x.x = (float)(x.x - cx); x.y = (float)(x.y - cy); x.z = (float)(x.z - cz);
    v.pos[g] = x;
  }
}

// Maxwell-Boltzmann momenta, centred per system (jax_md initialize_momenta):
// p = sqrt(m kT) xi, then p -= mean(p). One block per listed slot.
__global__ __launch_bounds__(kRedThreads) void k_init_momenta(DeviceView v, const int32_t* slot_list) {
  __shared__ double sh[kRedThreads];
  const int s = slot_list[blockIdx.x];
  const SlotConst& S = v.slots[s];
  double sx = 0, sy = 0, sz = 0;
  for (int i = threadIdx.x; i < S.n; i += kRedThreads) {
    const int g = S.a0 + i;
    const float3 xi = normal3(S.seed, 0u, i, 1u);
    const float a = S.sqrt_kT * v.sqrt_m[g];
    float4 p = v.mom[g];
    p.x = a * xi.x; p.y = a * xi.y; p.z = a * xi.z;
    v.mom[g] = p;
    v.atom_step[g] = 0u;
    sx += p.x; sy += p.y; sz += p.z;
  }
  const double mx = block_sum(sx, sh) / S.n;
  const double my = block_sum(sy, sh) / S.n;
  const double mz = block_sum(sz, sh) / S.n;
  if (S.n > 1) {
    for (int i = threadIdx.x; i < S.n; i += kRedThreads) {
      const int g = S.a0 + i;
      float4 p = v.mom[g];
      p.x = (float)(p.x - mx); p.y = (float)(p.y - my); p.z = (float)(p.z - mz);
      v.mom[g] = p;
    }
  }
}

// map[p] = arena index of packed atom p.
__global__ void k_copy_in_mom(DeviceView v, const float* src, const int32_t* map, int n) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int g = map[p];
  float4 m = v.mom[g];
  m.x = src[3 * p]; m.y = src[3 * p + 1]; m.z = src[3 * p + 2];
  v.mom[g] = m;
}

__global__ void k_copy_out(DeviceView v, float* pos, float* mom, float* frc, const int32_t* map, int n) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int g = map[p];
  if (pos) { const float4 a = v.pos[g]; pos[3 * p] = a.x; pos[3 * p + 1] = a.y; pos[3 * p + 2] = a.z; }
  if (mom) { const float4 a = v.mom[g]; mom[3 * p] = a.x; mom[3 * p + 1] = a.y; mom[3 * p + 2] = a.z; }
  if (frc) { const float4 a = v.force[g]; frc[3 * p] = a.x; frc[3 * p + 1] = a.y; frc[3 * p + 2] = a.z; }
}

static inline dim3 atom_grid(int n) { return dim3((n + 255) / 256); }

static inline dim3 tile_grid(int n_tiles) { return dim3((n_tiles + 3) / 4); }  // one wave per tile
static inline dim3 gather_grid(int n_tiles) { return dim3(n_tiles); }          // one block per tile

__device__ __forceinline__ int gather_wave() {
  return __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)));
}

__global__ __launch_bounds__(256) void k_tile_boxes(DeviceView v) {
  const int t = gather_wave();
  if (t >= v.n_tiles) return;
  tile_box_wave(v, t);
}

// The same, with the positions brought in from the caller's packed array on the
// way. With the forces and radii written by the gathers that form them and the
// bonded terms in the Born pass's launch, an evaluation takes 7 launches, with
// energies too in small systems, instead of 12, which bound these.
__global__ __launch_bounds__(256) void k_positions_in(DeviceView v, const float* packed) {
  const int t = gather_wave();
  if (t >= v.n_tiles) return;
  tile_box_wave(v, t, packed);
}

void launch_tile_boxes(const DeviceView& v, hipStream_t s) {
  if (v.n_tiles) hipLaunchKernelGGL(k_tile_boxes, tile_grid(v.n_tiles), dim3(256), 0, s, v);
}

void launch_born_gather(const DeviceView& v, float* packed_radii, hipStream_t s) {
  if (v.n_tiles) hipLaunchKernelGGL(k_born_gather, gather_grid(v.n_tiles), dim3(256), 0, s, v, packed_radii);
}
void launch_force_gather(const DeviceView& v, bool energy, hipStream_t s) {
  if (!v.n_tiles) return;
  if (energy)
    hipLaunchKernelGGL(k_force_gather<true>, gather_grid(v.n_tiles), dim3(256), 0, s, v);
  else
    hipLaunchKernelGGL(k_force_gather<false>, gather_grid(v.n_tiles), dim3(256), 0, s, v);
}
void launch_positions_in(const DeviceView& v, const float* packed, hipStream_t s) {
  if (v.n_tiles) hipLaunchKernelGGL(k_positions_in, tile_grid(v.n_tiles), dim3(256), 0, s, v, packed);
}
void launch_chain_gather(const DeviceView& v, int mode, float* packed_forces, hipStream_t s) {
  if (v.n_tiles) hipLaunchKernelGGL(k_chain_gather, gather_grid(v.n_tiles), dim3(256), 0, s, v, mode, packed_forces);
}
void launch_step_begin(const DeviceView& v, hipStream_t s) {
  if (v.atom_hw) hipLaunchKernelGGL(k_step_begin, atom_grid(v.atom_hw), dim3(256), 0, s, v);
}
void launch_energy_reduce(const DeviceView& v, const int32_t* ranges, int n_slots, double* out,
                          hipStream_t s) {
  if (n_slots) hipLaunchKernelGGL(k_energy_reduce, dim3(n_slots), dim3(kEnThreads), 0, s, v, ranges, out);
}
void launch_kinetic(const DeviceView& v, const int32_t* ranges, int n_slots, double* out, hipStream_t s) {
  if (n_slots) hipLaunchKernelGGL(k_kinetic, dim3(n_slots), dim3(kRedThreads), 0, s, v, ranges, out);
}
// One timestamp of the GPU's constant-rate wall clock, stored by lane 0 of a
// one-wave launch; graph dependencies order it between the passes around it.
__global__ void k_tick(unsigned long long* out) {
  const unsigned long long t = wall_clock64();
  if (threadIdx.x == 0) out[threadIdx.x] = t;
}

void launch_tick(unsigned long long* out, hipStream_t s) {
  hipLaunchKernelGGL(k_tick, dim3(1), dim3(64), 0, s, out);
}

void launch_recenter_com(const DeviceView& v, const int32_t* ranges, int n_slots, hipStream_t s) {
  if (n_slots) hipLaunchKernelGGL(k_recenter_com, dim3(n_slots), dim3(kRedThreads), 0, s, v, ranges);
}
void launch_init_momenta(const DeviceView& v, const int32_t* slot_list, int n, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_init_momenta, dim3(n), dim3(kRedThreads), 0, s, v, slot_list);
}
__global__ void k_fill_u32(uint32_t* dst, uint32_t value, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = value;
}

void launch_fill_u32(uint32_t* dst, uint32_t value, int n, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_fill_u32, atom_grid(n), dim3(256), 0, s, dst, value, n);
}
void launch_copy_in_momenta(const DeviceView& v, const float* src, const int32_t* map, int n,
                            hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_copy_in_mom, atom_grid(n), dim3(256), 0, s, v, src, map, n);
}
void launch_copy_out(const DeviceView& v, float* pos, float* mom, float* frc, const int32_t* map, int n,
                     hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_copy_out, atom_grid(n), dim3(256), 0, s, v, pos, mom, frc, map, n);
}

}  // namespace prx
