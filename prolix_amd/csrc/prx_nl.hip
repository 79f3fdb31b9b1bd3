// Neighbour lists of the gb_cut systems, built on the device at the start
// of an evaluation (after the tile boxes).
//
// The reference's neighbour-list path (physics/neighbor_list.py:155-172, a
// jax_md partition.neighbor_list with a Verlet skin; evaluated by
// generalized_born.py:266-415 and optimization.py:128-194, 299-357) keeps
// per-atom lists of partner atoms. Here the list is per 64-atom tile I: the
// atoms of the later tiles J > I that lie within cutoff + skin of tile I's
// bounding box, in increasing atom order. Pair kernels evaluate it in chunks
// of 64 listed atoms against the tile's 64 atoms with the per-pair cutoff
// test, so a chunk does the work of a tile pair, but only over atoms that can
// be in range: against whole tile pairs selected by box distance, this cuts
// the pair work of a 20,000-atom globule at a 20 A cutoff by ~40%.
//
// Two kernels; every list is a fixed function of the positions:
//   k_nl_check  per system with a skin: build this evaluation if forced or if an
//               atom moved more than skin / 2 since the last build (the
//               Verlet-skin rebuild rule of jax_md's neighbour list);
//   k_nl_rows   per tile I: for each J > I without exclusions a 64-bit mask of
//               the atoms of J within cutoff + skin of tile I's box, the prefix
//               counts over them, the list length and its entries. One block
//               keeps a row's masks and prefixes in LDS; with a wave per tile
//               pair for the masks and again for the entries, most of 48,828 waves
//               read a record and left (20,000 atoms: 4.6 + 9.1 + 5.6 + 6.8 us
//               a step; 10 steps 2,316 us then, 2,120 now).
// Tile pairs that hold exclusions stay ordinary items (their masks are 0).
#include "prx_nl_dev.h"

namespace prx {

namespace {

__device__ __forceinline__ int wave_index() {
  return __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)));
}

// One block per listed system.
__global__ __launch_bounds__(kNlThreads) void k_nl_check(DeviceView v, const int32_t* ranges) {
  nl_check_block(v, ranges, blockIdx.x);
}

// One block per tile. 10 steps of 20,000 atoms with 256, 512 and 1,024 threads:
// 2,194, 2,143 and 2,120 us (313 tiles: a row's box tests fit one round).
constexpr int kRowThreads = 1024;
__global__ __launch_bounds__(kRowThreads) void k_nl_rows(DeviceView v, int force) {
  nl_row_block<kRowThreads>(v, blockIdx.x, force);
}

// ---- dense atom lists (the drop-in neighbour-list object) -----------------
// Per atom i, every atom j != i closer than radius, in increasing j, in the
// (N, K) layout of a jax_md Dense neighbour list (sentinel N after the last
// entry); counts[i] = the true number, which may exceed K (overflow).

// Box of tile t of raw (N, 3) positions: (lo, hi) at boxes[2t], [2t + 1].
__global__ __launch_bounds__(kNlThreads) void k_dense_boxes(const float* pos, int n, float4* boxes) {
  const int t = wave_index();
  const int n_tiles = (n + kTile - 1) / kTile;
  if (t >= n_tiles) return;
  const int lane = threadIdx.x & 63;
  const int i = min(t * kTile + lane, n - 1);
  float lx = pos[3 * i], ly = pos[3 * i + 1], lz = pos[3 * i + 2];
  float hx = lx, hy = ly, hz = lz;
  for (int off = 32; off > 0; off >>= 1) {
    lx = fminf(lx, __shfl_xor(lx, off));
    ly = fminf(ly, __shfl_xor(ly, off));
    lz = fminf(lz, __shfl_xor(lz, off));
    hx = fmaxf(hx, __shfl_xor(hx, off));
    hy = fmaxf(hy, __shfl_xor(hy, off));
    hz = fmaxf(hz, __shfl_xor(hz, off));
  }
  if (lane == 0) boxes[2 * t] = make_float4(lx, ly, lz, 0.0f);
  if (lane == 1) boxes[2 * t + 1] = make_float4(hx, hy, hz, 0.0f);
}

// One wave per kListRows consecutive atoms. Its rows' own box is held against 64
// tile boxes at a time; for each tile in range lane = atom j, tested against every
// row, and a row's hits go out side by side at the row's count (the ballot's
// rank), so entries are in increasing j and stores and the sentinel fill are
// coalesced. The next tile's atoms are loaded while one is tested.
// One wave per 64 atoms, which walked every tile's atoms one by one with a
// store of four bytes per lane, left 313 waves on 1,024 SIMDs and was bound by its
// serial chain: 20,000 atoms at 9.5 A of a globule 304 us, of an assembly of
// domains 1,830 us. Rows per wave, us a list of the globule and a whole update of
// the assembly: 1: 25, 95; 2: 22, 88; 4: 25, 171; 8: 34 (fewer rows share a
// tile's load, more leave fewer waves and a larger box).
constexpr int kListRows = 2;

__global__ __launch_bounds__(kNlThreads) void k_dense_list(const float* pos, int n, float r2, int K, const float4* boxes,
                                                           int32_t* idx, int32_t* counts) {
  const int i0 = wave_index() * kListRows;
  if (i0 >= n) return;
  const int n_tiles = (n + kTile - 1) / kTile;
  const int lane = threadIdx.x & 63;
  float xi[kListRows], yi[kListRows], zi[kListRows];
  int cnt[kListRows];
#pragma unroll
  for (int r = 0; r < kListRows; ++r) {
    const int i = min(i0 + r, n - 1);
    xi[r] = pos[3 * (size_t)i]; yi[r] = pos[3 * (size_t)i + 1]; zi[r] = pos[3 * (size_t)i + 2];
    cnt[r] = 0;
  }
  float lx = xi[0], ly = yi[0], lz = zi[0], hx = xi[0], hy = yi[0], hz = zi[0];
#pragma unroll
  for (int r = 1; r < kListRows; ++r) {
    lx = fminf(lx, xi[r]); ly = fminf(ly, yi[r]); lz = fminf(lz, zi[r]);
    hx = fmaxf(hx, xi[r]); hy = fmaxf(hy, yi[r]); hz = fmaxf(hz, zi[r]);
  }
  for (int T0 = 0; T0 < n_tiles; T0 += 64) {
    const int T = min(T0 + lane, n_tiles - 1);
    const float4 lj = boxes[2 * T], hj = boxes[2 * T + 1];
    const float bx = fmaxf(0.0f, fmaxf(lj.x - hx, lx - hj.x));
    const float by = fmaxf(0.0f, fmaxf(lj.y - hy, ly - hj.y));
    const float bz = fmaxf(0.0f, fmaxf(lj.z - hz, lz - hj.z));
    unsigned long long near =
        __ballot(T0 + lane < n_tiles && !(bx * bx + by * by + bz * bz >= r2 * 1.00001f));
    if (near == 0ull) continue;
    int j = (T0 + __builtin_ctzll(near)) * kTile + lane;
    size_t at = 3 * (size_t)min(j, n - 1);
    float x = pos[at], y = pos[at + 1], z = pos[at + 2];
    while (near != 0ull) {
      const int jc = j;
      const float xc = x, yc = y, zc = z;
      near &= near - 1ull;
      if (near != 0ull) {
        j = (T0 + __builtin_ctzll(near)) * kTile + lane;
        at = 3 * (size_t)min(j, n - 1);
        x = pos[at]; y = pos[at + 1]; z = pos[at + 2];
      }
#pragma unroll
      for (int r = 0; r < kListRows; ++r) {
        const float dx = xc - xi[r], dy = yc - yi[r], dz = zc - zi[r];
        const bool hit = jc < n && jc != i0 + r && fmaf(dz, dz, fmaf(dy, dy, dx * dx)) < r2;
        const unsigned long long m = __ballot(hit);
        const int c = cnt[r] + __popcll(m & nl_below(lane));
        if (hit && i0 + r < n && c < K) idx[(size_t)(i0 + r) * K + c] = jc;
        cnt[r] += __popcll(m);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kListRows; ++r) {
    const int i = i0 + r;
    if (i >= n) break;
    if (lane == 0) counts[i] = cnt[r];
    for (int c = cnt[r] + lane; c < K; c += 64) idx[(size_t)i * K + c] = n;
  }
}

}  // namespace

void launch_dense_list(const float* pos, int n, float radius, int capacity, int32_t* idx, int32_t* counts,
                       float4* boxes, hipStream_t s) {
  if (n <= 0) return;
  const int n_tiles = (n + kTile - 1) / kTile;
  const int wpb = kNlThreads / 64;
  hipLaunchKernelGGL(k_dense_boxes, dim3((n_tiles + wpb - 1) / wpb), dim3(kNlThreads), 0, s, pos, n, boxes);
  const int per_block = wpb * kListRows;
  hipLaunchKernelGGL(k_dense_list, dim3((n + per_block - 1) / per_block), dim3(kNlThreads), 0, s, pos, n,
                     radius * radius, capacity, boxes, idx, counts);
}

void launch_nl_build(const DeviceView& v, const int32_t* slot_ranges, int n_slots, bool force, bool skins,
                     hipStream_t s) {
  if (n_slots <= 0 || v.n_tiles <= 0) return;
  if (!force && skins)
    hipLaunchKernelGGL(k_nl_check, dim3(n_slots), dim3(kNlThreads), 0, s, v, slot_ranges);
  hipLaunchKernelGGL(k_nl_rows, dim3(v.n_tiles), dim3(kRowThreads), 0, s, v, force ? 1 : 0);
}

}  // namespace prx
