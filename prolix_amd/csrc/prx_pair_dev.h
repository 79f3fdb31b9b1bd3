// Device code of the pair passes, shared by prx_pair.hip (one kernel per
// pass), prx_persist.hip and prx_fused.hip (every pass of a step in one kernel).
// BornPass, ForcePass and ChainPass are a wave's work on an item, or on a share
// of one ("Items to waves" below).
//
// A 64x64 item is 8x8 patches of 8x8 pairs. Lane l = 8 q + p takes the pair
// (row 8 b + q of tile I, column 8 a + p of tile J) of patch (b, a). Rows are
// read from LDS once per b and columns once per patch; the sums of the wave's
// eight columns (a = 0..7) stay in registers for the whole item, those of a row
// are added over the eight lanes p by DPP once per eight patches, and the
// columns' over q once at the end, so that no sum moves between lanes in the
// loop. Near pairs, which need square root, logarithm and clamps, are taken out
// of the loop: it marks their patches, and they are listed and evaluated 64 at
// a time behind it.
//
// What bounds it: VALU issue. gfx950 issues a plain FP32 instruction of one
// wave every 4.4 cycles and, with two or more waves per SIMD, one every 2.2
// cycles; transcendentals take 8.4, DPP operands 4.2, and the LDS of a CU
// takes 6 cycles per ds_bpermute and 8 per 16-byte read of a wave. One j atom
// per lane and iteration (64 rotations of the j sums through DPP or
// ds_bpermute, 1-2 LDS reads an iteration) bound the force pass by LDS: 40 of
// its 40 cycles per CU and iteration. A patch takes 26 (Born, average of its
// classes), 46 (force) and 37 (chain) VALU instructions, where an iteration
// took 40 to 50. 256 compact systems of 300 to 5,000 atoms, us a pass (Born, force,
// chain): 424, 655, 533 then, 373, 643, 501 now; one system of 2,500 atoms: 23.0,
// 18.9, 32.1 then, 10.4, 10.7, 12.6 now.
#pragma once

#include <type_traits>

#include "prx_common.h"
#include "prx_lanes_dev.h"
#include "prx_obc_farfield.h"

// Multiply-adds are fused only where the code says so: the sums of an item are the same
// on one, two and four waves only if each of their instances rounds alike, and left to
// itself the compiler fuses either product of a b + c d.
#pragma clang fp contract(off)

namespace prx {

__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float frsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ float flog2(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Orders this wave's LDS stores before its later LDS loads from other lanes.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Settings chosen by the autotuner (prolix_amd/tune.py) for this GPU; the
// defaults below apply to anything it leaves unset.
#include "prx_tuned.h"

// Unroll depth of the row loop (over b) of the three pair passes.
#ifndef PRX_UNROLL_BORN
#define PRX_UNROLL_BORN 1
#endif
#ifndef PRX_UNROLL_FORCE
#define PRX_UNROLL_FORCE 1
#endif
#ifndef PRX_UNROLL_CHAIN
#define PRX_UNROLL_CHAIN 1
#endif
// XCD-aware unit order (unit_id below).
#ifndef PRX_XCD_MAP
#define PRX_XCD_MAP 1
#endif
// Minimum waves per SIMD the compiler must fit the pair kernels' registers to
// (0: no constraint).
#ifndef PRX_MIN_WAVES
#define PRX_MIN_WAVES 0
#endif
#if PRX_MIN_WAVES > 0
#define PRX_OCCUPANCY __attribute__((amdgpu_waves_per_eu(PRX_MIN_WAVES)))
#define PRX_FORCE_OCCUPANCY(BLOCKS, ENERGY) PRX_OCCUPANCY
#else
#define PRX_OCCUPANCY
// The force pass: five waves per SIMD, without a spill (one system of 8,000 atoms 49.5
// us with four, 48.0); four with energies (five spill 15 registers: 256 systems of 300 to
// 5,000 atoms 1,950 us an evaluation, 2,065) and where a wave takes an item or a unit of any
// kind.
#define PRX_FORCE_OCCUPANCY(BLOCKS, ENERGY) \
  __attribute__((amdgpu_waves_per_eu(ENERGY || BLOCKS == 1 || BLOCKS == 0 ? 4 : 5)))
#endif
#define PRX_PRAGMA(x) _Pragma(#x)
#define PRX_UNROLL(n) PRX_PRAGMA(unroll n)

constexpr int kEdge = 8;          // edge of a patch
// Half h of an item's columns: the columns of patches a = h, h + 2, ... (neighbours in the
// sequence are near in a corner of the item, which left and right halves would give
// to one of them).
constexpr int kHalf = kEdge / 2;
// Half of column k of COLS (all, or those of one half).
template <int COLS>
__device__ constexpr int half_of(int k) { return COLS == kHalf ? 0 : k & 1; }

typedef float4 Tile4[kTile];
constexpr int kByte = sizeof(float4);

// Byte offset x, hidden from the optimiser and ready only once y is: the columns
// are read from LDS at such an offset, so that column a is read while column a - 1
// is evaluated. Left alone, the compiler reads all eight ahead of the row loop
// and keeps them, 8 x 8 to 12 registers that cost half the waves. (Of an index
// each read would shift a new one.)
__device__ __forceinline__ int after(int x, float y) {
  asm volatile("" : "+v"(x) : "v"(y));
  return x;
}
// Element at byte offset x of plane k of a staged tile.
__device__ __forceinline__ const float4& at_byte(const Tile4* t, int k, int x) {
  return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(t[k]) + x);
}

// Position of the lanes past the end of a ragged tile: so far away that every
// pair term underflows to zero or is multiplied by a zero parameter, and
// different for every lane, so that no such pair has r = 0.
__device__ __forceinline__ float4 pad_pos(int lane) { return make_float4(1e15f + 1e13f * (float)lane, 0.f, 0.f, 0.f); }

// ---------------------------------------------------------------------------
// Cross-lane sums
// ---------------------------------------------------------------------------
// Sum over the eight lanes p; every lane gets it.
__device__ __forceinline__ float sum_p(float x) {
  x += dpp<kDppHalfMirror>(x);
  x += dpp<kDppXor2>(x);
  x += dpp<kDppXor1>(x);
  return x;
}

// Sums over the eight lanes p of four values at once: lane p gets the
// sum of value comp_p(p). Each exchange halves the values a lane still
// carries: 4 DPP adds and 6 selects where four sums one by one take 12 DPP adds.
__device__ __forceinline__ int comp_p(int p) { return (p & 2) + ((p >> 2) & 1); }
__device__ __forceinline__ float sum_p4(float c0, float c1, float c2, float c3, int p) {
  const bool hi = (p & 4) != 0, mid = (p & 2) != 0;
  const float r0 = (hi ? c1 : c0) + dpp<kDppHalfMirror>(hi ? c0 : c1);
  const float r1 = (hi ? c3 : c2) + dpp<kDppHalfMirror>(hi ? c2 : c3);
  const float r = (mid ? r1 : r0) + dpp<kDppXor2>(mid ? r0 : r1);
  return r + dpp<kDppXor1>(r);
}
// Sums over the eight lane groups q of the eight columns v[a] of lane p: lane
// 8 q + p gets the sum of column a = q, which is atom (lane) of the tile.
__device__ __forceinline__ float sum_q(const float (&v)[kEdge], int lane) {
  float h[4], g[2];
#pragma unroll
  for (int a = 0; a < 4; ++a) h[a] = add_swap32(v[a], v[a + 4]);
#pragma unroll
  for (int a = 0; a < 2; ++a) g[a] = add_swap16(h[a], h[a + 2]);
  const bool odd = (lane & 8) != 0;
  return (odd ? g[1] : g[0]) + dpp<kDppRor8>(odd ? g[0] : g[1]);
}
// The same for the four columns of a half, in the same order of additions: lane l
// gets column l / 16 of them, atom half_col(l) of the half's 32.
__device__ __forceinline__ float sum_q(const float (&v)[kHalf], int) {
  const float g = add_swap16(add_swap32(v[0], v[2]), add_swap32(v[1], v[3]));
  return g + dpp<kDppRor8>(g);
}
__device__ __forceinline__ int half_col(int lane) { return kEdge * (lane >> 4) + (lane & 7); }
// Tile's atom i of the 32 of half h.
__device__ __forceinline__ int half_atom(int h, int i) { return 2 * (i & ~7) + kEdge * h + (i & 7); }

// The j atoms of an item: a tile (gj = j0 + lane), or for a chunk item of a
// neighbour list up to 64 listed atoms (gj = the lane's entry). nj = 0: an
// empty chunk (its row's list is shorter), which does nothing.
struct JSrc {
  int gj;  // this lane's j atom (clamped to the last valid one)
  int nj;  // j atoms of the item
};

__device__ __forceinline__ JSrc j_source(const DeviceView& v, const PairItem& it, int lane) {
  JSrc j;
  if (!item_is_chunk(it)) {
    j.nj = item_nj(it.meta);
    j.gj = it.j0 + min(lane, j.nj - 1);
    return j;
  }
  const int e0 = -1 - it.j0;
  j.nj = max(0, min(kTile, v.nl_count[it.ti] - (e0 - v.nl_row[it.ti].y)));
  j.gj = j.nj > 0 ? v.nl_entries[e0 + min(lane, j.nj - 1)] : 0;
  return j;
}

// ---------------------------------------------------------------------------
// OBC2 pair integral pieces
// ---------------------------------------------------------------------------

// Both directions of one pair share r and one reciprocal.
struct BornPair {
  float I1, I2;  // I(r; rho_i, s_j) and I(r; rho_j, s_i)
};

__device__ __forceinline__ BornPair born_pair(float r, float rinv, float rho_i, float s_i, float s_i2,
                                              float rho_j, float s_j, float s_j2) {
  const float U1 = r + s_j, U2 = r + s_i;
  const float L1 = fmaxf(fmaxf(rho_i, fabsf(r - s_j)), 1e-4f);
  const float L2 = fmaxf(fmaxf(rho_j, fabsf(r - s_i)), 1e-4f);
  const float U1c = fmaxf(U1, 1e-4f), U2c = fmaxf(U2, 1e-4f);
  const float p1 = L1 * U1c, p2 = L2 * U2c;
  const float inv = frcp(p1 * p2);
  const float ip1 = inv * p2, ip2 = inv * p1;
  const float iL1 = U1c * ip1, iU1 = L1 * ip1;
  const float iL2 = U2c * ip2, iU2 = L2 * ip2;
  const float rs = fminf(rinv, 1e4f);  // 1 / max(r, 1e-4)
  const float lg1 = flog2(L1 * iU1), lg2 = flog2(L2 * iU2);
  const float a1 = iL1 - iU1, a2 = iL2 - iU2;
  // 1/U^2 - 1/L^2 = -(1/L - 1/U)(1/L + 1/U)
  const float b1 = -a1 * (iL1 + iU1), b2 = -a2 * (iL2 + iU2);
  const float c1 = fmaf(-s_j2, rs, r), c2 = fmaf(-s_i2, rs, r);
  float I1 = fmaf(0.5f, a1, fmaf(0.25f * kLn2 * lg1, rs, 0.125f * c1 * b1));
  float I2 = fmaf(0.5f, a2, fmaf(0.25f * kLn2 * lg2, rs, 0.125f * c2 * b2));
  BornPair o;
  o.I1 = (U1 > rho_i) ? I1 : 0.0f;
  o.I2 = (U2 > rho_j) ? I2 : 0.0f;
  return o;
}

// dI/dr for one direction (rho = rho_i, s = sr_j), the derivative of born_pair's I.
__device__ __forceinline__ float born_dr(float r, float rs, float rho, float s, float s2) {
  const float dd = r - s;
  const float D = fabsf(dd);
  const bool useD = D > rho;
  const float L = useD ? D : rho;
  const float Lc = fmaxf(L, 1e-4f);
  float Lp = useD ? copysignf(1.0f, dd) : 0.0f;
  Lp = (L > 1e-4f) ? Lp : 0.0f;
  const float U = r + s;
  const float Uc = fmaxf(U, 1e-4f);
  const float Up = (U > 1e-4f) ? 1.0f : 0.0f;
  const float rp = (rs < 1e4f) ? 1.0f : 0.0f;
  const float inv = frcp(Lc * Uc);
  const float iL = Uc * inv, iU = Lc * inv;
  const float lg = flog2(Lc * iU) * kLn2;
  const float iL2 = iL * iL, iU2 = iU * iU;
  // Lp and Up are 0 or 1 in size, so these products are exact
  const float d1 = 0.5f * fmaf(Up, iU2, -(Lp * iL2));
  const float d2 = 0.25f * rs * fmaf(-(lg * rp), rs, fmaf(Lp, iL, -(Up * iU)));
  const float d3 = 0.125f * fmaf(s2 * rp, rs * rs, 1.0f) * (iU2 - iL2);
  const float d4 = 0.25f * fmaf(-s2, rs, r) * fmaf(Lp * iL2, iL, -(Up * iU2 * iU));
  // Every intermediate is finite (Lc, Uc >= 1e-4), so a 0/1 factor is exact
  // and keeps the wave free of a divergent branch.
  const float on = (U > rho) ? 1.0f : 0.0f;
  return on * (d1 + d2 + d3 + d4);
}

// Far field (r - s > rho and s <= r/2): L = r - s, U = r + s and
//   I = x^3 h(x^2) / (2r),  dI/dr = -x^3 k(x^2) / r^2,  x = s / r,
// with the polynomials of prx_obc_farfield.h. Same function as the direct
// formula, without its cancellation and without a transcendental.
__device__ __forceinline__ bool obc_far(float r, float rho, float s) {
  return (r - s > rho) && (s <= PRX_OBC_FAR_XMAX * r);
}

// How the Born and chain passes treat an item: every pair tested (kMixed), or
// every pair known to be in the far field (kFar) and at least 4, 6.5 or 14.5 s
// apart (kFar4, kFar3, kFar2: the polynomial's degree).
enum { kMixed = 0, kFar = 1, kFar4 = 2, kFar3 = 3, kFar2 = 4 };

// With u = 1/r^2 the far field is a polynomial in u whose coefficients belong
// to the descreening atom alone,
//   I = u^2 sum_k w_k u^k,           w_k = (s^3/3) s^(2k) h_k / h_0,
//   dI/dr = u^2 r^-1 sum_k w_k u^k,  w_k = -4 (s^3/3) s^(2k) k_k / k_0
// (h_0 = 2/3, k_0 = 4/3: the leading coefficient, all that counts far away, is s^3/3 of
// the atom's data, rounded once),
// so they are formed once per atom and item, and a direction of a pair costs
// one Horner chain in u and one fused multiply-add into its sum (against
// y = s^2 u, the chain in y, two products and an add: 5 against 8 operations
// a direction for the degree-4 fits).
template <int CLS>
struct BornW {
  static constexpr int N = (CLS == kFar2 ? kObcH2Deg : CLS == kFar3 ? kObcH3Deg : CLS == kFar4 ? kObcH4Deg : kObcHDeg) + 1;
  __device__ static constexpr float c(int k) {
    return (float)(1.5 * (CLS == kFar2 ? kObcH2[k] : CLS == kFar3 ? kObcH3[k] : CLS == kFar4 ? kObcH4[k] : kObcH[k]));
  }
};
template <int CLS>
struct ChainW {
  static constexpr int N = (CLS == kFar2 ? kObcK2Deg : CLS == kFar3 ? kObcK3Deg : CLS == kFar4 ? kObcK4Deg : kObcKDeg) + 1;
  __device__ static constexpr float c(int k) {
    return (float)(-3.0 * (CLS == kFar2 ? kObcK2[k] : CLS == kFar3 ? kObcK3[k] : CLS == kFar4 ? kObcK4[k] : kObcK[k]));
  }
};

// w[k] of one atom.
template <class W>
__device__ __forceinline__ void obc_weights(float s2, float s33, float (&w)[W::N]) {
  float m = s33;
#pragma unroll
  for (int k = 0; k < W::N; ++k) {
    w[k] = m * W::c(k);
    m *= s2;
  }
}

// sum_k w_k u^k / s33 for an atom whose weights are not formed: y = s^2 u.
template <class W>
__device__ __forceinline__ float obc_poly(float y) {
  float h = W::c(W::N - 1);
#pragma unroll
  for (int k = W::N - 2; k >= 0; --k) h = fmaf(h, y, W::c(k));
  return h;
}

template <int N>
__device__ __forceinline__ float horner(const float (&w)[N], float u) {
  float h = w[N - 1];
#pragma unroll
  for (int k = N - 2; k >= 0; --k) h = fmaf(h, u, w[k]);
  return h;
}

// ---------------------------------------------------------------------------
// Pass 1: Born sums
// ---------------------------------------------------------------------------

// LDS in float4: the rows (tile I) and columns (tile J) of an item, two per atom,
// and per wave a scratch list: 64 for the near pairs, later the sums that go to
// another wave ("Items to waves" below).
constexpr int kTilesLds = 4 * kTile;

// Scratch of a wave in float4: 64 for the list, later C sums of 64 rows (or, of a
// diagonal item, atoms) and of 32 columns.
template <int C>
constexpr int kObcScratch = C * (kTile + kTile / 2) / 4 > kTile ? C * (kTile + kTile / 2) / 4 : kTile;
// Memory of four waves that share an item: its tiles, per wave the lanes' sums of
// its four rows of patches (C sums each), per wave its scratch.
template <int C, int SCRATCH = kObcScratch<C>>
struct QuarterLds {
  static constexpr int kRowsLds = C * kHalf * 64 / 4;
  static constexpr int kSize = kTilesLds + 4 * (kRowsLds + SCRATCH);
  __device__ static __forceinline__ float* rows(float4* M, int k) {
    return reinterpret_cast<float*>(M + kTilesLds + k * kRowsLds);
  }
  __device__ static __forceinline__ float4* scratch(float4* M, int k) {
    return M + kTilesLds + 4 * kRowsLds + k * SCRATCH;
  }
};


// An atom of the Born pass. Short: the tiers of at most five coefficients,
// (x, y, z, w0), (w1, w2, w3, w4). The others keep (x, y, z, s^2), (s^3/3, rho,
// s, -): a row's weights are formed once per row of patches, a column takes
// obc_poly in y, two products more a pair than with weights but 16 bytes less
// per atom and read.
template <int CLS>
struct BornAtom {
  static constexpr int N = BornW<CLS>::N;
  static constexpr bool kShort = N <= 5;
  float x, y, z, s2, s33;
  float w[N];  // row, or short

  __device__ __forceinline__ static void stage(Tile4* t, int lane, const float4& p, const float4& b, float) {
    if constexpr (kShort) {
      float w[N];
      obc_weights<BornW<CLS>>(b.z, b.w, w);
      t[0][lane] = make_float4(p.x, p.y, p.z, w[0]);
      t[1][lane] = make_float4(w[1], w[2], N > 3 ? w[3 % N] : 0.0f, N > 4 ? w[4 % N] : 0.0f);
    } else {
      t[0][lane] = make_float4(p.x, p.y, p.z, b.z);
      t[1][lane] = make_float4(b.w, b.x, b.y, 0.0f);
    }
  }
  // row: with its weights
  __device__ __forceinline__ void read(const Tile4* t, int byte, bool row) {
    const float4 a = at_byte(t, 0, byte);
    x = a.x; y = a.y; z = a.z;
    if constexpr (kShort) {
      const float4 b = at_byte(t, 1, byte);
      w[0] = a.w; w[1] = b.x; w[2] = b.y;
      if constexpr (N > 3) w[3] = b.z;
      if constexpr (N > 4) w[4] = b.w;
    } else {
      s2 = a.w;
      s33 = at_byte(t, 1, byte).x;
      if (row) obc_weights<BornW<CLS>>(s2, s33, w);
    }
  }
  // sum_k w_k u^k
  __device__ __forceinline__ float sum(float u, bool row) const {
    if (kShort || row) return horner(w, u);
    return s33 * obc_poly<BornW<CLS>>(s2 * u);
  }
};

// The largest float below x > 0: r^2 < x is r^2 <= prev_below(x).
__device__ __forceinline__ float prev_below(float x) { return __int_as_float(__float_as_int(x) - 1); }

// The near pairs of a mixed item: those within lim2, of the patches marked in
// near (bit 8 b + a).
//
// Off the diagonal they are few (on proteins a tenth of the patches hold one,
// and three lanes of 64 in those: 20 to 40 pairs an item). They are listed first and
// evaluated 64 at a time, a pair per lane, by eval(row, col); then every lane adds,
// in list order, the terms of its row 8 p + q and of its column my_col by
// add_row(half, terms, mine) and add_col(terms, mine), factors of 1 or 0. Terms that are
// not finite (two atoms at one point), which a factor of 0 would hand to every row and
// column, are added by selects behind their batch instead (selects for every term:
// 1.4% of the chain pass of 256 systems of 300 to 5,000 atoms).
// HALVES: near holds patches of both halves, whose row sums are kept apart: those of
// half 1 are listed from the other end of the scratch and evaluated in the lanes
// behind the first's, from a multiple of kBatch on, so that the loops that add
// need no test (a branch per entry on its half: 1.5 us of 9.3 of the Born pass of 138
// atoms, whose waves wait for the scalar unit).
template <bool HALVES, class Eval, class Row, class Col>
__device__ __forceinline__ void near_list(const Tile4* ti, const Tile4* tj, unsigned long long near, int lane,
                                          int my_col, bool cut, float lim2, float4* scratch, Eval&& eval,
                                          Row&& add_row, Col&& add_col) {
  constexpr int kBatch = 4;  // entries read before any is added
  constexpr int kList = 128;
  const int p = lane & 7, q = lane >> 3, my_row = kEdge * p + q;
  unsigned short* const list = reinterpret_cast<unsigned short*>(scratch);
  int count[2] = {0, 0};
  for (;;) {
    while (near != 0 && count[0] + count[1] < 64) {
      const int k = __builtin_ctzll(near), row = (k & 56) + q, col = kEdge * (k & 7) + p;
      near &= near - 1;
      const float4 a = ti[0][row], b = tj[0][col];
      const float dx = b.x - a.x, dy = b.y - a.y, dz = b.z - a.z;
      const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
      const bool on = cut ? r2 <= lim2 : !(r2 > lim2);
      const unsigned long long m = __ballot(on);
      const bool back = HALVES && (k & 1);
      int at = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
      at = back ? kList - 1 - count[1] - at : count[0] + at;
      if (on) list[at] = (unsigned short)(row << 6 | col);
      count[0] += back ? 0 : __popcll(m);
      count[1] += back ? __popcll(m) : 0;
    }
    if (count[0] + count[1] == 0) break;
    wave_lds_sync();
    const int n0 = min(count[0], 64), b1 = (n0 + kBatch - 1) & -kBatch;  // lanes of half 0, first lane of half 1
    const int n1 = HALVES ? min(count[1], 64 - b1) : 0;
    const bool on = lane < n0 || (HALVES && lane >= b1 && lane < b1 + n1);
    int e = list[HALVES && lane >= b1 ? kList - 1 - (lane - b1) : min(lane, max(n0 - 1, 0))];
    int rest0 = 0, rest1 = 0;
    if (HALVES) {
      rest0 = list[min(64 + lane, kList - 1)];
      rest1 = list[max(kList - 1 - n1 - lane, 0)];
      e = on ? e : 0;
    } else {
      rest0 = list[64 + lane];
    }
    wave_lds_sync();
    const float3 t = eval(e >> 6, e & 63);
    const bool sound = fabsf(t.x) + fabsf(t.y) + fabsf(t.z) < INFINITY;
    scratch[lane] = make_float4(sound ? t.x : 0.0f, sound ? t.y : 0.0f, sound ? t.z : 0.0f,
                                __int_as_float(on ? e : -1));
    wave_lds_sync();
    const auto add = [&](int from, int to, auto half) {
      for (int k = from; k < to; k += kBatch) {
        float4 c[kBatch];
#pragma unroll
        for (int m = 0; m < kBatch; ++m) c[m] = scratch[k + m];
#pragma unroll
        for (int m = 0; m < kBatch; ++m) {
          const int ce = __float_as_int(c[m].w);
          add_row(half, c[m], (ce >> 6) == my_row ? 1.0f : 0.0f);
          add_col(c[m], ce >= 0 && (ce & 63) == my_col ? 1.0f : 0.0f);
        }
      }
    };
    add(0, n0, std::integral_constant<int, 0>());
    if (HALVES) add(b1, b1 + n1, std::integral_constant<int, 1>());
    for (unsigned long long m = __ballot(on && !sound); m != 0; m &= m - 1) {
      const int k = __builtin_ctzll(m), ce = __builtin_amdgcn_readlane(e, k);
      const float4 c = make_float4(__shfl(t.x, k), __shfl(t.y, k), __shfl(t.z, k), 0.0f);
      const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
      add_row(std::integral_constant<int, 0>(), (ce >> 6) == my_row ? c : zero, 1.0f);
      add_col((ce & 63) == my_col ? c : zero, 1.0f);
    }
    wave_lds_sync();
    count[0] -= n0;
    count[1] -= n1;
    if (lane < count[0]) list[lane] = (unsigned short)rest0;
    if (HALVES && lane < count[1]) list[kList - 1 - lane] = (unsigned short)rest1;
  }
}

// On the diagonal a fifth of the pairs are near (14 to 20 per atom): a lane walks
// those of its own atom with the rows of share s, on both sides of the diagonal, so
// nothing is summed across lanes. The even and the odd ones of them are summed
// apart, by add(atom, near, on, sum, sum) two at a time (one is a chain of dependent
// steps), so that an atom can have a lane of its own (atom = lane) or with SPLIT two: lanes
// l and l + 32 take the even and the odd near atoms of atom l of half h and get its sum.
template <bool SPLIT, int C, class Add>
__device__ __forceinline__ void near_diag(const Tile4* t, int lane, int ni, int s, int nsub, int h, bool cut,
                                          float lim2, Add&& add, float (&sum)[C]) {
  const int second = SPLIT ? lane >> 5 : 0, atom = SPLIT ? half_atom(h, lane & 31) : lane;
  const float4 me = t[0][atom];
  unsigned long long near = 0;
  // two lanes test every other row of patches each
  for (int b = s + nsub * second; kEdge * b < ni; b += SPLIT ? 2 * nsub : nsub) {
    unsigned bits = 0;
#pragma unroll
    for (int k = 0; k < kEdge; ++k) {
      const float4 o = t[0][kEdge * b + k];
      // the sign of the difference as in the pair loop: later atom minus earlier
      const float dx = o.x - me.x, dy = o.y - me.y, dz = o.z - me.z;
      const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
      const bool on = (cut ? r2 <= lim2 : !(r2 > lim2)) && kEdge * b + k != atom && kEdge * b + k < ni;
      bits |= on ? 1u << k : 0u;
    }
    near |= (unsigned long long)bits << (kEdge * b);
  }
  if (SPLIT) {
    const unsigned x = (unsigned)near, y = (unsigned)(near >> 32);
    const auto lo = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(y, y, false, false);
    near = (unsigned long long)(hi[0] | hi[1]) << 32 | (lo[0] | lo[1]);
    if (second) near &= near - 1;
  }
  if (atom >= ni) near = 0;
  float even[C] = {}, odd[C] = {};
  while (__any(near != 0)) {
    int o[2];
    bool on[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      on[k] = near != 0;
      o[k] = on[k] ? __builtin_ctzll(near) : atom;
      near &= near - 1;
      if (SPLIT) near &= near - 1;  // the other lane's
    }
    add(atom, o, on, even, SPLIT ? even : odd);
  }
#pragma unroll
  for (int c = 0; c < C; ++c) sum[c] += SPLIT ? add_swap32(even[c], even[c]) : even[c] + odd[c];
}

// I(r; rho_i, s_j) alone, for a near or a far pair.
__device__ __forceinline__ float born_one(float r2, float rho_i, float s_j, float s2_j, float s33_j) {
  const float rinv = frsq(r2), r = r2 * rinv, u = rinv * rinv;
  const float U = r + s_j;
  const float L = fmaxf(fmaxf(rho_i, fabsf(r - s_j)), 1e-4f), Uc = fmaxf(U, 1e-4f);
  const float inv = frcp(L * Uc), iL = Uc * inv, iU = L * inv;
  const float rs = fminf(rinv, 1e4f);
  const float a = iL - iU, b = -a * (iL + iU), c = fmaf(-s2_j, rs, r);
  const float I = fmaf(0.5f, a, fmaf(0.25f * kLn2 * flog2(L * iU), rs, 0.125f * c * b));
  return obc_far(r, rho_i, s_j) ? (u * u) * (s33_j * obc_poly<BornW<kMixed>>(s2_j * u)) : (U > rho_i ? I : 0.0f);
}

// Near pairs of two atoms o of a diagonal item (near_diag).
__device__ __forceinline__ void born_near_diag(const Tile4* t, int atom, const int (&o)[2], const bool (&on)[2],
                                               float (&even)[1], float (&odd)[1]) {
  const float4 me = t[0][atom];
  const float rhoi = t[1][atom].y;
  float I[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float4 a = t[0][o[k]], b = t[1][o[k]];
    const float dx = a.x - me.x, dy = a.y - me.y, dz = a.z - me.z;
    I[k] = born_one(fmaf(dx, dx, fmaf(dy, dy, dz * dz)), rhoi, b.z, a.w, b.x);
  }
  even[0] += on[0] ? I[0] : 0.0f;
  odd[0] += on[1] ? I[1] : 0.0f;
}

// Terms of a near pair off the diagonal: x to the row, y to the column.
__device__ __forceinline__ float3 born_near_pair(const Tile4* ti, const Tile4* tj, int row, int col) {
  const float4 ai = ti[0][row], bi = ti[1][row], aj = tj[0][col], bj = tj[1][col];
  const float rhoi = bi.y, si = bi.z, rhoj = bj.y, sj = bj.z;
  const float dx = aj.x - ai.x, dy = aj.y - ai.y, dz = aj.z - ai.z;
  const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
  const float rinv = frsq(r2);
  const float u = rinv * rinv, u2 = u * u, r = r2 * rinv;
  const BornPair bp = born_pair(r, rinv, rhoi, si, ai.w, rhoj, sj, aj.w);
  const float I1 = obc_far(r, rhoi, sj) ? u2 * (bj.x * obc_poly<BornW<kMixed>>(aj.w * u)) : bp.I1;
  const float I2 = obc_far(r, rhoj, si) ? u2 * (bi.x * obc_poly<BornW<kMixed>>(ai.w * u)) : bp.I2;
  return make_float3(I1, I2, 0.0f);
}

// The atoms of an item's tiles (or of one of them), loaded together: lane = atom.
struct ItemAtoms {
  float4 pi, bi, pj, bj;
  float ci, cj;
};
template <bool CHAIN>
__device__ __forceinline__ ItemAtoms load_atoms(const DeviceView& v, const PairItem& it, const JSrc& js, int lane,
                                                bool rows, bool cols) {
  const int gi = it.i0 + min(lane, item_ni(it.meta) - 1), gj = js.gj;
  ItemAtoms t;
  t.ci = t.cj = 0.0f;
  if (rows) {
    t.pi = v.pos[gi]; t.bi = v.born4[gi];
    if (CHAIN) t.ci = v.gb4[gi].w;
  }
  if (cols) {
    t.pj = v.pos[gj]; t.bj = v.born4[gj];
    if (CHAIN) t.cj = v.gb4[gj].w;
  }
  return t;
}
// Lanes past the end of a ragged tile: far away, and without any term.
__device__ __forceinline__ void pad_atoms(ItemAtoms& t, int lane, int ni, int nj) {
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  if (lane >= ni) { t.pi = pad_pos(lane); t.bi = zero; t.ci = 0.0f; }
  if (lane >= nj) { t.pj = pad_pos(lane); t.bj = zero; t.cj = 0.0f; }
}

// The far pairs of the rows b = sub, sub + nsub, ... of an item with COLS columns
// of patches: all eight (rows: lane 8 q + p gets the sum of row 8 p + q) or those of
// half h (the lanes' row sums go to t, [row of the share][lane]). A row's sum is that
// of its half 0 plus that of its half 1, lane by lane, so both ways give the same. cols: the columns' sums over these rows, as sum_q leaves them.
// CUT: pairs with r^2 >= cut2 add nothing. FULL: both tiles hold 64 atoms.
// thr2: above it every pair of the item is in the far field; a mixed item
// adds only the pairs above it here and marks the patches of the others in
// near, so that the loop has no branch and the registers of the far field alone.
template <int CLS, bool DIAG, bool CUT, bool FULL, int COLS>
__device__ __forceinline__ void born_tile(const float4* L, int ni, int nj, int lane, float cut2, float thr2, int sub,
                                          int nsub, int h, float* t, float (&rows)[1], float (&cols)[1],
                                          unsigned long long& near) {
  const Tile4* ti = reinterpret_cast<const Tile4*>(L);
  const Tile4* tj = ti + 2;
  const int p = lane & 7, q = lane >> 3;
  float accj[COLS] = {};
  BornAtom<CLS> half_cols[kHalf];  // of half h, kept over the rows
  if (COLS == kHalf)
#pragma unroll
    for (int k = 0; k < kHalf; ++k) half_cols[k].read(tj, kByte * (p + kEdge * (2 * k + h)), false);
  const int nb = FULL ? kEdge : (ni + kEdge - 1) / kEdge, na = FULL ? kEdge : (nj + kEdge - 1) / kEdge;
  PRX_UNROLL(PRX_UNROLL_BORN)
  for (int b = sub; b < nb; b += nsub) {
    BornAtom<CLS> i;
    float half[2] = {};
    i.read(ti, kByte * (kEdge * b + q), true);
    unsigned marks = 0;
    int col = kByte * p;
#pragma unroll
    for (int k = 0; k < COLS; ++k) {
      const int a = COLS == kHalf ? 2 * k + h : k;
      if (!FULL && a >= na) continue;
      if (DIAG && a < b) continue;
      float& acci = half[half_of<COLS>(k)];
      BornAtom<CLS> j;
      if constexpr (COLS == kHalf) {
        j = half_cols[k];
      } else {
        col = after(col, k < 2 ? acci : accj[k - 2]);
        j.read(tj, col + kByte * kEdge * k, false);
      }
      const float dx = j.x - i.x, dy = j.y - i.y, dz = j.z - i.z;
      float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
      if (DIAG && a == b) r2 = p > q ? r2 : 1e30f;  // each unordered pair once: no term at 1e15 A
      bool on = true;
      if (CUT) on = r2 < cut2;
      if (CLS == kMixed) {
        const bool close = !(r2 > thr2);
        if (!DIAG) marks |= (__ballot(on && close) != 0 ? 1u : 0u) << a;
        on = on && !close;
      }
      float u = frcp(r2);
      if (CUT || CLS == kMixed) u = on ? u : 0.0f;
      const float u2 = u * u;
      acci = fmaf(u2, j.sum(u, false), acci);
      accj[k] = fmaf(u2, i.sum(u, true), accj[k]);
    }
    if constexpr (COLS == kHalf) {
      t[(b >> 1) * 64 + lane] = half[0];
    } else {
      const float r = sum_p(half[0] + half[1]);
      rows[0] = p == b ? r : rows[0];
    }
    if (CLS == kMixed && !DIAG) near |= (unsigned long long)marks << (kEdge * b);
  }
  cols[0] = sum_q(accj, lane);
}

// Class bits of an item from its tiles' bounding boxes (wave-uniform). The
// far-field tier needs the box distance above every pair's threshold,
// max(s_j + rho_i, s_i + rho_j, 2 s) over the two tiles, with a 1e-4
// relative margin on the squared distance; the finer tiers also need it above
// 4, 6.5 and 14.5 s.
__device__ __forceinline__ int classify(const DeviceView& v, const SlotConst& S, const PairItem& it, float& thr2) {
  const int tI = it.ti, tJ = it.tj;
  const float4 li = v.tbox[2 * tI], hi = v.tbox[2 * tI + 1];
  const float4 lj = v.tbox[2 * tJ], hj = v.tbox[2 * tJ + 1];
  const float gx = fmaxf(0.0f, fmaxf(lj.x - hi.x, li.x - hj.x));
  const float gy = fmaxf(0.0f, fmaxf(lj.y - hi.y, li.y - hj.y));
  const float gz = fmaxf(0.0f, fmaxf(lj.z - hi.z, li.z - hj.z));
  const float ex = fmaxf(hj.x - li.x, hi.x - lj.x);
  const float ey = fmaxf(hj.y - li.y, hi.y - lj.y);
  const float ez = fmaxf(hj.z - li.z, hi.z - lj.z);
  const float dmin2 = gx * gx + gy * gy + gz * gz;
  const float dmax2 = ex * ex + ey * ey + ez * ez;
  const float thr = fmaxf(fmaxf(hj.w + li.w, hi.w + lj.w), fmaxf(hi.w, hj.w) * (1.0f / PRX_OBC_FAR_XMAX));
  thr2 = thr * thr * 1.0001f;
  const float smax = fmaxf(hi.w, hj.w), d2 = dmin2 * (1.0f / 1.0001f);
  const float t4 = smax * (1.0f / PRX_OBC_FAR4_XMAX), t3 = smax * (1.0f / PRX_OBC_FAR3_XMAX);
  const float t2 = smax * (1.0f / PRX_OBC_FAR2_XMAX);
  int tier = kMixed;
  if (tI != tJ && dmin2 > thr2) tier = d2 > t2 * t2 ? kFar2 : d2 > t3 * t3 ? kFar3 : d2 > t4 * t4 ? kFar4 : kFar;
  int cls = tier << kClsTierShift;
  if (S.cutoff2 > 0.0f) {
    if (dmin2 >= S.cutoff2 * 1.00001f)
      cls |= kClsFar;
    else if (!(dmax2 < S.cutoff2 * 0.99999f))
      cls |= kClsStraddle;
  }
  return cls;
}

// Class of a chunk item: every listed pair may straddle the cutoff; the OBC2
// far-field bit comes from the i tile's box and the box of the chunk's j
// atoms (a wave reduction over the lanes' atoms), as for a tile pair.
__device__ __forceinline__ int classify_chunk(const DeviceView& v, const PairItem& it, const float4& p,
                                              const float4& b, float& thr2) {
  float lx = p.x, ly = p.y, lz = p.z, hx = p.x, hy = p.y, hz = p.z, mr = b.x, ms = b.y;
  for (int off = 32; off > 0; off >>= 1) {
    lx = fminf(lx, __shfl_xor(lx, off));
    ly = fminf(ly, __shfl_xor(ly, off));
    lz = fminf(lz, __shfl_xor(lz, off));
    hx = fmaxf(hx, __shfl_xor(hx, off));
    hy = fmaxf(hy, __shfl_xor(hy, off));
    hz = fmaxf(hz, __shfl_xor(hz, off));
    mr = fmaxf(mr, __shfl_xor(mr, off));
    ms = fmaxf(ms, __shfl_xor(ms, off));
  }
  const float4 li = v.tbox[2 * it.ti], hi = v.tbox[2 * it.ti + 1];
  const float gx = fmaxf(0.0f, fmaxf(lx - hi.x, li.x - hx));
  const float gy = fmaxf(0.0f, fmaxf(ly - hi.y, li.y - hy));
  const float gz = fmaxf(0.0f, fmaxf(lz - hi.z, li.z - hz));
  const float dmin2 = gx * gx + gy * gy + gz * gz;
  const float thr = fmaxf(fmaxf(ms + li.w, hi.w + mr), fmaxf(hi.w, ms) * (1.0f / PRX_OBC_FAR_XMAX));
  thr2 = thr * thr * 1.0001f;
  const float t4 = fmaxf(hi.w, ms) * (1.0f / PRX_OBC_FAR4_XMAX);
  const int tier = !(dmin2 > thr2) ? kMixed : (dmin2 * (1.0f / 1.0001f) > t4 * t4 ? kFar4 : kFar);
  return kClsStraddle | (tier << kClsTierShift);
}

// A system at its step limit, in a step graph (DeviceView::skip_done).
__device__ __forceinline__ bool skip_item(const DeviceView& v, const SlotConst& S, const PairItem& it) {
  return v.skip_done && S.step_limit != 0u && slot_done(S, v.atom_step[it.i0]);
}

// item_cls holds an item's class (low bits) and, in the others, the Born
// pass's far-field threshold thr^2 as a float rounded up: a pair with r^2 above
// it is in the far field in both directions.
__device__ __forceinline__ int pack_cls(int cls, float thr2) {
  return ((__float_as_int(thr2) + kClsMask) & ~kClsMask) | cls;
}
__device__ __forceinline__ float cls_thr2(int packed) { return __int_as_float(packed & ~kClsMask); }

// Runs f.run<CLS, DIAG, CUT, FULL>() for an item of class tier. Ragged and
// cut items take the degree-4 polynomials at best: they are few, and every
// variant costs instruction cache.
template <class F>
__device__ __forceinline__ void by_class(int tier, bool diag, bool cut, bool full, F&& f) {
  if (diag) {
    if (cut)
      f.template run<kMixed, true, true, false>();
    else
      f.template run<kMixed, true, false, false>();
  } else if (cut) {
    if (tier >= kFar4)
      f.template run<kFar4, false, true, false>();
    else if (tier == kFar)
      f.template run<kFar, false, true, false>();
    else
      f.template run<kMixed, false, true, false>();
  } else if (!full) {
    if (tier >= kFar4)
      f.template run<kFar4, false, false, false>();
    else if (tier == kFar)
      f.template run<kFar, false, false, false>();
    else
      f.template run<kMixed, false, false, false>();
  } else {
    if (tier == kFar2)
      f.template run<kFar2, false, false, true>();
    else if (tier == kFar3)
      f.template run<kFar3, false, false, true>();
    else if (tier == kFar4)
      f.template run<kFar4, false, false, true>();
    else if (tier == kFar)
      f.template run<kFar, false, false, true>();
    else
      f.template run<kMixed, false, false, true>();
  }
}

// An item's rows and/or columns into LDS in the form of its class (template
// ATOM); done with before the pairs, so that the loaded atoms hold no registers
// there.
template <template <int> class ATOM>
struct StageRun {
  const ItemAtoms& t;
  int lane;
  bool rows, cols;
  float4* L;
  template <int CLS, bool DIAG, bool CUT, bool FULL>
  __device__ __forceinline__ void run() {
    Tile4* ti = reinterpret_cast<Tile4*>(L);
    if (rows) ATOM<CLS>::stage(ti, lane, t.pi, t.bi, t.ci);
    if (cols) ATOM<CLS>::stage(ti + 2, lane, t.pj, t.bj, t.cj);
  }
};

template <int COLS>
struct BornRun {
  const float4* L;
  int ni, nj, lane;
  float cut2, thr2;
  int sub, nsub, h;
  float* t;
  float rows[1], cols[1];
  unsigned long long near;
  template <int CLS, bool DIAG, bool CUT, bool FULL>
  __device__ __forceinline__ void run() {
    born_tile<CLS, DIAG, CUT, FULL, COLS>(L, ni, nj, lane, cut2, thr2, sub, nsub, h, t, rows, cols, near);
  }
};

// C sums per row and per column of one item: Born (C = 1) and chain (C = 3).
template <int C>
__device__ __forceinline__ void put_sums(float* at, int stride, int lane, const float (&v)[C]) {
#pragma unroll
  for (int c = 0; c < C; ++c) at[c * stride + lane] = v[c];
}
template <int C>
__device__ __forceinline__ void add_sums(float (&v)[C], const float (&o)[C]) {
#pragma unroll
  for (int c = 0; c < C; ++c) v[c] += o[c];
}
template <int C>
struct ObcSum {
  float v[C] = {};
  __device__ __forceinline__ void add(const ObcSum& o) { add_sums(v, o.v); }
  __device__ __forceinline__ void to_lds(float4* at, int lane) const {
    put_sums(reinterpret_cast<float*>(at), kTile, lane, v);
  }
  __device__ __forceinline__ void from_lds(const float4* at, int lane) {
#pragma unroll
    for (int c = 0; c < C; ++c) v[c] = reinterpret_cast<const float*>(at)[c * kTile + lane];
  }
};

// The Born and the chain pass over one item; Self has stage(), which prepares it
// (rows and/or cols: which of its tiles this wave brings into LDS; false: the item has
// no work, and no partials), the pass's run, near-pair functions and partials.
template <class Self, int C>
struct ObcPass {
  typedef ObcSum<C> Sum;
  typedef QuarterLds<C> Quarter;
  static constexpr int kLaneEnergies = 0;
  int w, lane, ni, nj, tier, nsub;
  float cut2, thr2, lim2;
  bool diag, full, cut;

  // Near pairs of a diagonal item: sums of its atoms.
  template <bool SPLIT>
  __device__ __forceinline__ void near_atoms(const float4* L, int s, int h, float (&sum)[C]) const {
    const Tile4* t = reinterpret_cast<const Tile4*>(L);
    near_diag<SPLIT>(
        t, lane, ni, s, nsub, h, cut, lim2,
        [&](int atom, const int (&o)[2], const bool (&on)[2], float (&even)[C], float (&odd)[C]) {
          Self::near_two(t, atom, o, on, even, odd);
        },
        sum);
  }

  // Near pairs off the diagonal of one share: added to its rows' and its columns' sums.
  template <bool HALVES>
  __device__ __forceinline__ void near_pairs(const float4* L, float4* scratch, unsigned long long near, int my_col,
                                             float (&rows)[C], float (&cols)[C]) const {
    const Tile4* ti = reinterpret_cast<const Tile4*>(L);
    const Tile4* tj = ti + 2;
    float n0[C] = {}, n1[C] = {}, m[C] = {};
    near_list<HALVES>(
        ti, tj, near, lane, my_col, cut, lim2, scratch,
        [&](int row, int col) { return Self::near_pair(ti, tj, row, col); },
        [&](auto half, const float4& c, float mine) { Self::add_row(decltype(half)::value ? n1 : n0, c, mine); },
        [&](const float4& c, float mine) { Self::add_col(m, c, mine); });
    add_sums(rows, n0);
    add_sums(rows, n1);
    add_sums(cols, m);
  }

  // Share s: its rows' sums (zero in the other's lanes) and its columns' (lane = atom),
  // far and then near. scratch: this wave's own.
  __device__ __forceinline__ void share(int s, const float4* L, float4* scratch, float (&rows)[C],
                                        float (&cols)[C]) const {
    typename Self::template Run<kEdge> f{L, ni, nj, lane, cut2, thr2, s, nsub, 0, nullptr, {}, {}, 0};
    by_class(tier, diag, cut, full, f);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      rows[c] = f.rows[c];
      cols[c] = f.cols[c];
    }
    if (diag) {
      float d[C] = {};
      near_atoms<false>(L, s, 0, d);
      add_sums(cols, d);
    } else if (f.near != 0) {
      near_pairs<true>(L, scratch, f.near, lane, rows, cols);
    }
  }

  // Share s0, or with LOOP the shares s0 .. s1 - 1: stores the rows' sums and
  // returns the columns', share 0's plus share 1's.
  template <bool LOOP>
  __device__ __forceinline__ Sum run(const DeviceView& v, int s0, int s1, const float4* L, float4* scratch) const {
    const int p = lane & 7, q = lane >> 3, mine = p & (nsub - 1);
    Sum sum;
    if constexpr (LOOP) {
      float rows[C] = {};
#pragma unroll 1
      for (int s = s0; s < s1; ++s) {
        float r[C], c[C];
        share(s, L, scratch, r, c);
        add_sums(rows, r);
        add_sums(sum.v, c);
      }
      if (mine >= s0 && mine < s1) Self::put(v, w, 0, kEdge * p + q, rows);
    } else {
      float rows[C];
      share(s0, L, scratch, rows, sum.v);
      if (mine == s0) Self::put(v, w, 0, kEdge * p + q, rows);
    }
    return sum;
  }

  // The item by four waves: wave k = 2 s + h takes share s of the rows and half h
  // of the columns. M: the group's memory (QuarterLds).
  __device__ __forceinline__ Sum quarter(int k, float4* M) const {
    typedef Quarter Q;
    const int s = k >> 1, h = k & 1;
    float4* const scratch = Q::scratch(M, k);
    typename Self::template Run<kHalf> f{M, ni, nj, lane, cut2, thr2, s, nsub, h, Q::rows(M, k), {}, {}, 0};
    by_class(tier, diag, cut, full, f);
    Sum sum;
    add_sums(sum.v, f.cols);
    if (diag) {
      float d[C] = {};
      near_atoms<true>(M, s, h, d);
      put_sums(reinterpret_cast<float*>(scratch), kTile, lane, d);
      wave_lds_sync();
#pragma unroll
      for (int c = 0; c < C; ++c) sum.v[c] += reinterpret_cast<const float*>(scratch)[c * kTile + half_col(lane)];
    } else {
      float near[C] = {};  // of the rows
      if (f.near != 0)
        near_pairs<false>(M, scratch, f.near, half_atom(h, half_col(lane)), near, sum.v);
      put_sums(reinterpret_cast<float*>(scratch), kTile, lane, near);
    }
    if (s == 1 && (lane & 8) == 0)
      put_sums(reinterpret_cast<float*>(scratch) + C * kTile, kTile / 2, half_col(lane), sum.v);
    return sum;
  }

  // Behind the barrier: wave k finishes two of its share's rows of patches, the
  // waves of share 0 the columns of their half.
  __device__ __forceinline__ void finish(const DeviceView& v, int k, float4* M, Sum& sum) const {
    typedef Quarter Q;
    const int s = k >> 1, h = k & 1, p = lane & 7, q = lane >> 3;
    float rows[C] = {};
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int i = 2 * h + n, b = s + 2 * i;
      if (kEdge * b >= ni) break;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int at = (c * kHalf + i) * 64 + lane;
        const float r = sum_p(Q::rows(M, 2 * s)[at] + Q::rows(M, 2 * s + 1)[at]);
        rows[c] = p == b ? r : rows[c];
      }
    }
    const float* const n0 = reinterpret_cast<const float*>(Q::scratch(M, 2 * s));
    const float* const n1 = reinterpret_cast<const float*>(Q::scratch(M, 2 * s + 1));
    if (!diag)
#pragma unroll
      for (int c = 0; c < C; ++c) rows[c] = (rows[c] + n0[c * kTile + lane]) + n1[c * kTile + lane];
    if ((p & 1) == s && (p >> 2) == h) Self::put(v, w, 0, kEdge * p + q, rows);
    if (s != 0) return;
    const int half = half_col(lane);
    const float* const c1 = reinterpret_cast<const float*>(Q::scratch(M, 2 + h)) + C * kTile;
    float cols[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      cols[c] = sum.v[c] + c1[c * (kTile / 2) + half];
    }
    if ((lane & 8) == 0) Self::put(v, w, 1, half_atom(h, half), cols);
  }

  __device__ __forceinline__ void store(const DeviceView& v, const Sum& s) const { Self::put(v, w, 1, lane, s.v); }
};

struct BornPass : ObcPass<BornPass, 1> {
  template <int COLS>
  using Run = BornRun<COLS>;
  static constexpr int kRows = 1, kScratch = kObcScratch<1>;

  __device__ __forceinline__ static float3 near_pair(const Tile4* ti, const Tile4* tj, int row, int col) {
    return born_near_pair(ti, tj, row, col);
  }
  __device__ __forceinline__ static void add_row(float (&n)[1], const float4& c, float mine) {
    n[0] = fmaf(mine, c.x, n[0]);
  }
  __device__ __forceinline__ static void add_col(float (&m)[1], const float4& c, float mine) {
    m[0] = fmaf(mine, c.y, m[0]);
  }
  __device__ __forceinline__ static void near_two(const Tile4* t, int atom, const int (&o)[2], const bool (&on)[2],
                                                  float (&even)[1], float (&odd)[1]) {
    born_near_diag(t, atom, o, on, even, odd);
  }
  __device__ __forceinline__ static void put(const DeviceView& v, int w, int side, int at, const float (&x)[1]) {
    part1(v, w, side)[at] = x[0];
  }

  __device__ __forceinline__ bool stage(const DeviceView& v, int w_, const PairItem& it, bool rows, bool cols,
                                        float4* L) {
    w = w_;
    lane = threadIdx.x & 63;
    const SlotConst& S = v.slots[item_slot(it.meta)];
    if (skip_item(v, S, it)) return false;
    const bool chunk = item_is_chunk(it);
    const JSrc js = j_source(v, it, lane);
    ItemAtoms t = load_atoms<false>(v, it, js, lane, rows, cols || chunk);
    diag = (item_flags(it.meta) & kFlagDiag) != 0;
    ni = item_ni(it.meta);
    nj = js.nj;
    full = ni == kTile && nj == kTile;
    nsub = it.nsub;
    thr2 = 0.0f;
    int cls;
    if (chunk) {  // neighbour-list chunk: always with the cutoff test
      if (nj == 0) {
        if (lane == 0 && rows) v.item_cls[w] = kClsFar;
        return false;
      }
      cls = classify_chunk(v, it, t.pj, t.bj, thr2);
    } else {
      cls = classify(v, S, it, thr2);
    }
    if (lane == 0 && rows) v.item_cls[w] = pack_cls(cls, thr2);
    const int ccut = cls & kClsCutMask;
    if (S.gb_cut && ccut == kClsFar) return false;  // no partials: the gathers skip this item
    cut = S.gb_cut && ccut == kClsStraddle;
    cut2 = S.cutoff2;
    lim2 = cut ? fminf(thr2, prev_below(cut2)) : thr2;
    tier = cls >> kClsTierShift;
    if (!full) pad_atoms(t, lane, ni, nj);
    StageRun<BornAtom> put{t, lane, rows, cols, L};
    by_class(tier, diag, cut, full, put);
    return true;
  }
};

// ---------------------------------------------------------------------------
// Pass 2: GB + Coulomb + LJ
// ---------------------------------------------------------------------------

// Column sums of a share: force, sum of g B_i of lane's atom; e: an energy
// summed over the wave, GB in lanes 0-15, Coulomb in 32-47, LJ in the others
// (sum_energies).
template <bool ENERGY>
struct ForceSum {
  float x = 0.0f, y = 0.0f, z = 0.0f, g = 0.0f;
  double e = 0.0;
  __device__ __forceinline__ void add(const ForceSum& o) {
    x += o.x; y += o.y; z += o.z; g += o.g;
    if (ENERGY) e += o.e;
  }
  __device__ __forceinline__ void put_energies(const DeviceView& v, int w, int lane) const {
    if (ENERGY && lane < 48 && (lane & 15) == 0) v.e_items[(size_t)w * 3 + (lane == 0 ? 0 : (lane == 32 ? 1 : 2))] = e;
  }
  __device__ __forceinline__ void to_lds(float4* at, int lane, int atom) const {
    at[atom] = make_float4(x, y, z, g);
    if (ENERGY && (lane & 15) == 0) reinterpret_cast<double*>(at + kTile)[lane >> 4] = e;
  }
  __device__ __forceinline__ void to_lds(float4* at, int lane) const { to_lds(at, lane, lane); }
  __device__ __forceinline__ double energy_from_lds(const float4* at, int lane) const {
    return ENERGY ? reinterpret_cast<const double*>(at + kTile)[lane >> 4] : 0.0;
  }
  __device__ __forceinline__ void from_lds(const float4* at, int lane, int atom) {
    const float4 f = at[atom];
    x = f.x; y = f.y; z = f.z; g = f.w;
    e = energy_from_lds(at, lane);
  }
  __device__ __forceinline__ void from_lds(const float4* at, int lane) { from_lds(at, lane, lane); }
};

// Three doubles summed over the wave, in the lanes of ForceSum::e: each
// exchange puts two values' sums into the halves of one register.
__device__ __forceinline__ double sum_energies(double gb, double cl, double lj) {
  double e = add_swap<false>(add_swap<true>(gb, cl), add_swap<true>(lj, lj));
  e += dpp<kDppRor8>(e);
  e += dpp<kDppRor8 - 4>(e);
  e += dpp<kDppRor8 - 6>(e);
  return e + dpp<kDppRor8 - 7>(e);
}

// Row sums of a patch row, from its lanes p.
__device__ __forceinline__ void put_force_row(float* side0, int row, int p, float x, float y, float z, float db) {
  const float s = sum_p4(x, y, z, -0.5f * db, p);
  if ((p & 1) == 0) side0[row * 4 + comp_p(p)] = s;
}

// Three energies of this lane's pairs added to its sums in LDS.
__device__ __forceinline__ void add_energies(double* en, int lane, const double (&e)[3]) {
#pragma unroll
  for (int c = 0; c < 3; ++c) en[c * 64 + lane] += e[c];
}

// What the pass takes from its system's constants and its item.
struct ForceConst {
  float kc, gb2, cut2;  // cut2 > 0: the test r^2 < cut2 per pair
  bool gb_cut;          // of GB too
  float ev[4], ee[4];   // scales by exclusion class
  const ulonglong2* excl;  // the rows' exclusion masks, or nullptr
};

// LJC = false: GB only (items entirely beyond the LJ/Coulomb cutoff). GEN:
// ragged tiles, exclusions, and with cut2 > 0 the test r^2 < cut2 per pair, on
// LJ/Coulomb and, if gb_cut, on GB too. COLS, h and t as in born_tile. The energies too
// are summed by halves, a row of patches at a time: with all eight columns the sums of
// both halves wait in LDS (en: [half][term][lane]), where in registers they cost a
// wave per SIMD, and a row takes the columns of half 0 first.
template <bool GEN, bool DIAG, bool ENERGY, bool LJC, int COLS>
__device__ __forceinline__ void force_tile(const ForceConst& S, int ni, int nj, int lane, float* side0, int sub,
                                           int nsub, int h, float* t, const float4* L, double* en, ForceSum<ENERGY>& out) {
  const Tile4* ti = reinterpret_cast<const Tile4*>(L);
  const Tile4* tj = ti + 2;
  const float kc = S.kc, gb2 = S.gb2, cut2 = S.cut2;
  const bool has_cut = GEN && cut2 > 0.0f, gb_cut = S.gb_cut;
  const bool has_excl = GEN && LJC && S.excl != nullptr;
  const int p = lane & 7, q = lane >> 3;
  float fxj[COLS] = {}, fyj[COLS] = {}, fzj[COLS] = {}, dbj[COLS] = {};
  constexpr int kTerms = 3;
  double e[kTerms] = {};  // GB, Coulomb, LJ / 4
  if (ENERGY && COLS == kEdge)
#pragma unroll
    for (int k = 0; k < 2 * kTerms; ++k) en[k * 64 + lane] = 0.0;
  const int nb = GEN ? (ni + kEdge - 1) / kEdge : kEdge, na = GEN ? (nj + kEdge - 1) / kEdge : kEdge;
  ulonglong2 next = {};  // a short loop waits for these loads: half an item's are issued a row ahead
  float4 half_a[kHalf], half_b[kHalf];  // columns of half h, kept over the rows
  if (COLS == kHalf)
#pragma unroll
    for (int k = 0; k < kHalf; ++k) {
      half_a[k] = tj[0][p + kEdge * (2 * k + h)];
      half_b[k] = tj[1][p + kEdge * (2 * k + h)];
    }
  PRX_UNROLL(PRX_UNROLL_FORCE)
  for (int b = sub; b < nb; b += nsub) {
    const int row = kEdge * b + q;
    const float4 ia = ti[0][row], ib = ti[1][row];
    const float q_kc = kc * ia.w, q_gb = gb2 * ia.w;
    float fx[COLS / kHalf] = {}, fy[COLS / kHalf] = {}, fz[COLS / kHalf] = {}, db[COLS / kHalf] = {};
    unsigned long long m0 = 0, m1 = 0;  // the row's exclusion classes, column p of each patch at bit 8 a
    if (has_excl) {
      if (COLS == kEdge || b == sub) next = S.excl[row];
      m0 = next.x >> p;
      m1 = next.y >> p;
      if (COLS == kHalf && b + nsub < nb) next = S.excl[row + kEdge * nsub];
    }
    int col = kByte * p;
    double er[kTerms] = {};  // of the row's columns of one half
#pragma unroll
    for (int n = 0; n < COLS; ++n) {
      // place n's column: with energies half 0's before half 1's
      const auto place = [](int n) { return ENERGY && COLS == kEdge ? 2 * (n % kHalf) + n / kHalf : n; };
      const int k = place(n);
      if (ENERGY && COLS == kEdge && n == kHalf) {
        add_energies(en, lane, er);
#pragma unroll
        for (int c = 0; c < kTerms; ++c) er[c] = 0.0;
      }
      const int a = COLS == kHalf ? 2 * k + h : k;
      if (GEN && a >= na) continue;
      if (DIAG && a < b) continue;
      const int o = half_of<COLS>(k);
      float &fxi = fx[o], &fyi = fy[o], &fzi = fz[o], &dbi = db[o];
      float4 ja, jb;
      if constexpr (COLS == kHalf) {
        ja = half_a[k];
        jb = half_b[k];
      } else {
        col = after(col, n < 2 ? fxi : fxj[place(n - 2)]);
        ja = at_byte(tj, 0, col + kByte * kEdge * k);
        jb = at_byte(tj, 1, col + kByte * kEdge * k);
      }
      const float dx = ja.x - ia.x, dy = ja.y - ia.y, dz = ja.z - ia.z;
      float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
      const bool once = !DIAG || a != b || p > q;  // each unordered pair once
      if (DIAG && a == b) r2 = once ? r2 : 1e30f;
      const bool in = !has_cut || r2 < cut2;
      if (has_cut && gb_cut && !__any(in)) continue;
      float lc = 0.0f, rinv2 = 0.0f;  // -dE/dr r of Coulomb + LJ
      if (LJC && (!has_cut || __any(in))) {
        const float rinv = frsq(r2);
        rinv2 = rinv * rinv;
        float ec = (q_kc * ja.w) * rinv;
        const float sg = ib.x + jb.x;
        const float ep = ib.y * jb.y;
        const float s2 = sg * sg * rinv2;
        const float s6 = s2 * s2 * s2;
        float el = ep * fmaf(s6, s6, -s6);  // / 4
        const float es6 = ep * s6, f6 = fmaf(48.0f, s6, -24.0f);
        float fl = es6 * f6;
        if (GEN) {
          if (has_excl) {
            const unsigned e0 = (unsigned)(m0 >> (kEdge * a)) & 1u, e1 = (unsigned)(m1 >> (kEdge * a)) & 1u;
            const unsigned cls = e0 | (e1 << 1);
            if (__any(cls != 0u)) {
              const float sv = cls == 0 ? 1.0f : (cls == 1 ? S.ev[1] : (cls == 2 ? S.ev[2] : S.ev[3]));
              const float se = cls == 0 ? 1.0f : (cls == 1 ? S.ee[1] : (cls == 2 ? S.ee[2] : S.ee[3]));
              const bool some = sv != 0.0f || se != 0.0f;
              ec = some ? ec * se : 0.0f;
              el = some ? el * sv : 0.0f;
              fl = some ? fl * sv : 0.0f;
            }
          }
          if (has_cut) {
            ec = in ? ec : 0.0f;
            el = in ? el : 0.0f;
            fl = in ? fl : 0.0f;
          }
        }
        if (ENERGY) {
          er[1] += once ? (double)ec : 0.0;
          er[2] += once ? (double)el : 0.0;
        }
        lc = GEN ? ec + fl : fmaf(es6, f6, ec);
      }
      // GB over every pair
      const float BB = ib.z * jb.z;
      const float x = r2 * (ib.w * jb.w);  // r^2 log2(e) / (4 B_i B_j)
      const float ex = fexp2(-x);
      const float f2 = fmaf(BB, ex, r2);
      const float finv = frsq(f2);
      const float eg = (q_gb * ja.w) * finv;
      const float tg = eg * (finv * finv);  // gb2 qq / f^3
      const float te = tg * ex;
      float fgb = fmaf(-0.25f, te, tg);    // -dE/dr / r
      float g = te * fmaf(x, kLn2, 1.0f);  // dE/dB_i = -g B_j / 2, dE/dB_j = -g B_i / 2
      if (GEN && has_cut && gb_cut) {
        fgb = in ? fgb : 0.0f;
        g = in ? g : 0.0f;
        if (ENERGY) er[0] += in && once ? (double)eg : 0.0;
      } else if (ENERGY) {
        er[0] += once ? (double)eg : 0.0;
      }
      const float fr = LJC ? fmaf(lc, rinv2, fgb) : fgb;
      // F_i = -fr * (x_j - x_i)
      fxi = fmaf(-fr, dx, fxi); fyi = fmaf(-fr, dy, fyi); fzi = fmaf(-fr, dz, fzi);
      dbi = fmaf(g, jb.z, dbi);
      fxj[k] = fmaf(fr, dx, fxj[k]); fyj[k] = fmaf(fr, dy, fyj[k]); fzj[k] = fmaf(fr, dz, fzj[k]);
      dbj[k] = fmaf(g, ib.z, dbj[k]);
    }
    if (ENERGY && COLS == kEdge) add_energies(en + kTerms * 64, lane, er);
    if (ENERGY && COLS == kHalf)
#pragma unroll
      for (int c = 0; c < kTerms; ++c) e[c] += er[c];
    if constexpr (COLS == kHalf) {
      reinterpret_cast<float4*>(t)[(b >> 1) * 64 + lane] = make_float4(fx[0], fy[0], fz[0], db[0]);
    } else {
      put_force_row(side0, row, p, fx[0] + fx[1], fy[0] + fy[1], fz[0] + fz[1], db[0] + db[1]);
    }
  }
  out.x = sum_q(fxj, lane);
  out.y = sum_q(fyj, lane);
  out.z = sum_q(fzj, lane);
  out.g = -0.5f * sum_q(dbj, lane);
  if (ENERGY && COLS == kHalf) out.e = sum_energies(e[0], e[1], 4.0 * e[2]);
  if (ENERGY && COLS == kEdge) {
    const double* e1 = en + kTerms * 64;
    out.e = sum_energies(en[lane], en[64 + lane], 4.0 * en[128 + lane]);
    out.e += sum_energies(e1[lane], e1[64 + lane], 4.0 * e1[128 + lane]);
  }
}

// The force pass over one item (as BornPass).
template <bool ENERGY>
struct ForcePass {
  typedef ForceSum<ENERGY> Sum;
  static constexpr int kRows = 4, kScratch = kTile;               // columns
  static constexpr int kLaneEnergies = ENERGY ? 2 * 3 * 64 / 2 : 0;  // the lanes' energies by half, later the wave's
  typedef QuarterLds<kRows, kScratch + 2> Quarter;                   // with the wave's energies
  int w, lane, ni, nj, cls, nsub, flags;
  ForceConst K;
  float* side0;
  bool full;

  __device__ __forceinline__ bool stage(const DeviceView& v, int w_, const PairItem& it, bool rows, bool cols,
                                        float4* L) {
    w = w_;
    lane = threadIdx.x & 63;
    const SlotConst& S = v.slots[item_slot(it.meta)];
    if (!ENERGY && skip_item(v, S, it)) return false;
    cls = S.cutoff2 > 0.0f ? (v.item_cls[w] & kClsCutMask) : kClsNear;
    if (cls == kClsFar && S.gb_cut) {
      if (ENERGY && lane < 3 && rows) v.e_items[(size_t)w * 3 + lane] = 0.0;
      return false;
    }
    const JSrc js = j_source(v, it, lane);
    ni = item_ni(it.meta);
    nj = js.nj;
    full = ni == kTile && nj == kTile;
    nsub = it.nsub;
    flags = item_flags(it.meta);
    side0 = reinterpret_cast<float*>(part4(v, w, 0));
    K.kc = S.k_coulomb;
    K.gb2 = S.gb2;
    K.cut2 = cls == kClsStraddle ? S.cutoff2 : 0.0f;
    K.gb_cut = S.gb_cut != 0;
    K.excl = it.excl >= 0 ? reinterpret_cast<const ulonglong2*>(v.excl_masks) + (size_t)it.excl * kTile : nullptr;
    for (int k = 1; k < 4; ++k) {
      K.ev[k] = S.excl_v[k];
      K.ee[k] = S.excl_e[k];
    }
    // (x, y, z, q), (sigma/2, sqrt(eps), B, a) of the rows and the columns
    const int gi = it.i0 + min(lane, ni - 1), gj = js.gj;
    float4 pi, ci, bi, pj, cj, bj;
    if (rows) { pi = v.pos[gi]; ci = v.nb4[gi]; bi = v.gb4[gi]; }
    if (cols) { pj = v.pos[gj]; cj = v.nb4[gj]; bj = v.gb4[gj]; }
    Tile4* t = reinterpret_cast<Tile4*>(L);
    // past the end of a ragged tile: no charge, no well depth, B = 1 and next to no
    // exponent (0 times the r^2 of an atom at infinity would not be a number)
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f), one = make_float4(1.f, 1e-30f, 0.f, 0.f);
    if (rows) {
      if (!full && lane >= ni) { pi = pad_pos(lane); ci = zero; bi = one; }
      t[0][lane] = make_float4(pi.x, pi.y, pi.z, ci.x);
      t[1][lane] = make_float4(ci.y, ci.z, bi.x, bi.y);
    }
    if (cols) {
      if (!full && lane >= nj) { pj = pad_pos(lane); cj = zero; bj = one; }
      t[2][lane] = make_float4(pj.x, pj.y, pj.z, cj.x);
      t[3][lane] = make_float4(cj.y, cj.z, bj.x, bj.y);
    }
    return true;
  }

  template <int COLS>
  __device__ __forceinline__ Sum share(int sub, int h, float* t, const float4* L, double* en) const {
    Sum f;
    if (cls == kClsFar) {  // GB over every pair, nothing else (a far item is never diagonal)
      if (full)
        force_tile<false, false, ENERGY, false, COLS>(K, ni, nj, lane, side0, sub, nsub, h, t, L, en, f);
      else
        force_tile<true, false, ENERGY, false, COLS>(K, ni, nj, lane, side0, sub, nsub, h, t, L, en, f);
    } else if (flags & kFlagDiag) {
      force_tile<true, true, ENERGY, true, COLS>(K, ni, nj, lane, side0, sub, nsub, h, t, L, en, f);
    } else if (full && !(flags & kFlagExcl) && K.cut2 == 0.0f) {
      force_tile<false, false, ENERGY, true, COLS>(K, ni, nj, lane, side0, sub, nsub, h, t, L, en, f);
    } else {
      force_tile<true, false, ENERGY, true, COLS>(K, ni, nj, lane, side0, sub, nsub, h, t, L, en, f);
    }
    return f;
  }

  // As in ObcPass.
  template <bool LOOP>
  __device__ __forceinline__ Sum run(const DeviceView&, int s0, int s1, const float4* L, float4* scratch) const {
    double* const en = reinterpret_cast<double*>(scratch + kScratch);
    if constexpr (!LOOP) return share<kEdge>(s0, 0, nullptr, L, en);
    Sum sum;
#pragma unroll 1
    for (int sub = s0; sub < s1; ++sub) sum.add(share<kEdge>(sub, 0, nullptr, L, en));
    return sum;
  }

  __device__ __forceinline__ Sum quarter(int k, float4* M) const {
    const Sum sum = share<kHalf>(k >> 1, k & 1, Quarter::rows(M, k), M, nullptr);
    if (k != 0) sum.to_lds(Quarter::scratch(M, k), lane, half_col(lane));
    return sum;
  }

  __device__ __forceinline__ void finish(const DeviceView& v, int k, float4* M, Sum& sum) const {
    const int s = k >> 1, h = k & 1, p = lane & 7, q = lane >> 3;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const int i = 2 * h + n, b = s + 2 * i;
      if (kEdge * b >= ni) break;
      const float4 x = reinterpret_cast<const float4*>(Quarter::rows(M, 2 * s))[i * 64 + lane];
      const float4 y = reinterpret_cast<const float4*>(Quarter::rows(M, 2 * s + 1))[i * 64 + lane];
      put_force_row(side0, kEdge * b + q, p, x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w);
    }
    if (s != 0) return;
    const int half = half_col(lane);
    Sum o;
    o.from_lds(Quarter::scratch(M, 2 + h), lane, half);
    if (ENERGY && h == 0) {
      sum.e += sum.energy_from_lds(Quarter::scratch(M, 1), lane);
      o.e += o.energy_from_lds(Quarter::scratch(M, 3), lane);
    }
    sum.add(o);
    if ((lane & 8) == 0) part4(v, w, 1)[half_atom(h, half)] = make_float4(sum.x, sum.y, sum.z, sum.g);
    if (h == 0) sum.put_energies(v, w, lane);
  }

  __device__ __forceinline__ void store(const DeviceView& v, const Sum& s) const {
    part4(v, w, 1)[lane] = make_float4(s.x, s.y, s.z, s.g);
    s.put_energies(v, w, lane);
  }
};

// ---------------------------------------------------------------------------
// Pass 3: chain rule through the Born radii
// ---------------------------------------------------------------------------

// An atom of the chain pass: short (x, y, z, c), (w0, w1, w2, w3), else
// (x, y, z, c), (s^2, s^3/3, rho, s), as BornAtom.
template <int CLS>
struct ChainAtom {
  static constexpr bool kShort = ChainW<CLS>::N <= 4;
  float x, y, z, c, s2, s33;
  float w[ChainW<CLS>::N];

  __device__ __forceinline__ static void stage(Tile4* t, int lane, const float4& p, const float4& b, float c) {
    t[0][lane] = make_float4(p.x, p.y, p.z, c);
    if constexpr (kShort) {
      float w[ChainW<CLS>::N];
      obc_weights<ChainW<CLS>>(b.z, b.w, w);
      t[1][lane] = make_float4(w[0], w[1], w[2], ChainW<CLS>::N > 3 ? w[3 % ChainW<CLS>::N] : 0.0f);
    } else {
      t[1][lane] = make_float4(b.z, b.w, b.x, b.y);
    }
  }
  __device__ __forceinline__ void read(const Tile4* t, int byte, bool row) {
    const float4 a = at_byte(t, 0, byte);
    x = a.x; y = a.y; z = a.z; c = a.w;
    if constexpr (kShort) {
      const float4 b = at_byte(t, 1, byte);
      w[0] = b.x; w[1] = b.y; w[2] = b.z;
      if constexpr (ChainW<CLS>::N > 3) w[3] = b.w;
    } else {
      const float2 b = *reinterpret_cast<const float2*>(&at_byte(t, 1, byte));
      s2 = b.x;
      s33 = b.y;
      if (row) obc_weights<ChainW<CLS>>(s2, s33, w);
    }
  }
  // sum_k w_k u^k
  __device__ __forceinline__ float sum(float u, bool row) const {
    if (kShort || row) return horner(w, u);
    return s33 * obc_poly<ChainW<CLS>>(s2 * u);
  }
};

// gsc of a near or far pair (chain_tile); a = (x, y, z, c), b = (s^2, s^3/3, rho, s).
__device__ __forceinline__ float chain_one(float r2, float ci, const float4& bi, float cj, const float4& bj) {
  const float rinv = frsq(r2), u = rinv * rinv, u2r = u * u * rinv, r = r2 * rinv, rs = fminf(rinv, 1e4f);
  const float d1 = obc_far(r, bi.z, bj.w) ? u2r * (bj.y * obc_poly<ChainW<kMixed>>(bj.x * u))
                                          : born_dr(r, rs, bi.z, bj.w, bj.x);
  const float d2 = obc_far(r, bj.z, bi.w) ? u2r * (bi.y * obc_poly<ChainW<kMixed>>(bi.x * u))
                                          : born_dr(r, rs, bj.z, bi.w, bi.x);
  return fmaf(ci, d1, cj * d2) * rinv;
}

__device__ __forceinline__ void chain_near_diag(const Tile4* t, int atom, const int (&o)[2], const bool (&on)[2],
                                                float (&even)[3], float (&odd)[3]) {
  const float4 me = t[0][atom], mb = t[1][atom];
  float g[2], dx[2], dy[2], dz[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float4 a = t[0][o[k]], b = t[1][o[k]];
    dx[k] = a.x - me.x; dy[k] = a.y - me.y; dz[k] = a.z - me.z;
    const float r2 = fmaf(dx[k], dx[k], fmaf(dy[k], dy[k], dz[k] * dz[k]));
    g[k] = chain_one(on[k] ? r2 : 1.0f, me.w, mb, a.w, b);
  }
  const float f = on[0] ? g[0] : 0.0f, e = on[1] ? g[1] : 0.0f;
  even[0] = fmaf(f, dx[0], even[0]); even[1] = fmaf(f, dy[0], even[1]); even[2] = fmaf(f, dz[0], even[2]);
  odd[0] = fmaf(e, dx[1], odd[0]); odd[1] = fmaf(e, dy[1], odd[1]); odd[2] = fmaf(e, dz[1], odd[2]);
}

// Force of a near pair off the diagonal on its row atom.
__device__ __forceinline__ float3 chain_near_pair(const Tile4* ti, const Tile4* tj, int row, int col) {
  const float4 ai = ti[0][row], bi = ti[1][row], aj = tj[0][col], bj = tj[1][col];
  const float dx = aj.x - ai.x, dy = aj.y - ai.y, dz = aj.z - ai.z;
  const float gsc = chain_one(fmaf(dx, dx, fmaf(dy, dy, dz * dz)), ai.w, bi, aj.w, bj);
  return make_float3(gsc * dx, gsc * dy, gsc * dz);
}

// As born_tile. Per pair: F_i = gsc (x_j - x_i), gsc = (c_i dI(rho_i, s_j)/dr +
// c_j dI(rho_j, s_i)/dr) / r, in the far field u^3 (c_i P_j(u) + c_j P_i(u)).
template <int CLS, bool DIAG, bool CUT, bool FULL, int COLS>
__device__ __forceinline__ void chain_tile(const float4* L, int ni, int nj, int lane, float cut2, float thr2, int sub,
                                           int nsub, int h, float* t, float (&rows)[3], float (&cols)[3],
                                           unsigned long long& near) {
  const Tile4* ti = reinterpret_cast<const Tile4*>(L);
  const Tile4* tj = ti + 2;
  const int p = lane & 7, q = lane >> 3;
  float fxj[COLS] = {}, fyj[COLS] = {}, fzj[COLS] = {};
  ChainAtom<CLS> half_cols[kHalf];
  if (COLS == kHalf)
#pragma unroll
    for (int k = 0; k < kHalf; ++k) half_cols[k].read(tj, kByte * (p + kEdge * (2 * k + h)), false);
  const int nb = FULL ? kEdge : (ni + kEdge - 1) / kEdge, na = FULL ? kEdge : (nj + kEdge - 1) / kEdge;
  PRX_UNROLL(PRX_UNROLL_CHAIN)
  for (int b = sub; b < nb; b += nsub) {
    ChainAtom<CLS> i;
    float fx[2] = {}, fy[2] = {}, fz[2] = {};
    i.read(ti, kByte * (kEdge * b + q), true);
    unsigned marks = 0;
    int col = kByte * p;
#pragma unroll
    for (int k = 0; k < COLS; ++k) {
      const int a = COLS == kHalf ? 2 * k + h : k;
      if (!FULL && a >= na) continue;
      if (DIAG && a < b) continue;
      float &fxi = fx[half_of<COLS>(k)], &fyi = fy[half_of<COLS>(k)], &fzi = fz[half_of<COLS>(k)];
      ChainAtom<CLS> j;
      if constexpr (COLS == kHalf) {
        j = half_cols[k];
      } else {
        col = after(col, k < 2 ? fxi : fxj[k - 2]);
        j.read(tj, col + kByte * kEdge * k, false);
      }
      const float dx = j.x - i.x, dy = j.y - i.y, dz = j.z - i.z;
      float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
      if (DIAG && a == b) r2 = p > q ? r2 : 1e30f;
      bool on = true;
      if (CUT) on = r2 < cut2;
      if (CLS == kMixed) {
        const bool close = !(r2 > thr2);
        if (!DIAG) marks |= (__ballot(on && close) != 0 ? 1u : 0u) << a;
        on = on && !close;
      }
      float u = frcp(r2);
      if (CUT || CLS == kMixed) u = on ? u : 0.0f;
      const float gsc = (u * u * u) * fmaf(i.c, j.sum(u, false), j.c * i.sum(u, true));
      fxi = fmaf(gsc, dx, fxi); fyi = fmaf(gsc, dy, fyi); fzi = fmaf(gsc, dz, fzi);
      fxj[k] = fmaf(-gsc, dx, fxj[k]); fyj[k] = fmaf(-gsc, dy, fyj[k]); fzj[k] = fmaf(-gsc, dz, fzj[k]);
    }
    if constexpr (COLS == kHalf) {
      const float x[3] = {fx[0], fy[0], fz[0]};
#pragma unroll
      for (int c = 0; c < 3; ++c) t[(c * kHalf + (b >> 1)) * 64 + lane] = x[c];
    } else {
      const float x = sum_p(fx[0] + fx[1]), y = sum_p(fy[0] + fy[1]), z = sum_p(fz[0] + fz[1]);
      rows[0] = p == b ? x : rows[0]; rows[1] = p == b ? y : rows[1]; rows[2] = p == b ? z : rows[2];
    }
    if (CLS == kMixed && !DIAG) near |= (unsigned long long)marks << (kEdge * b);
  }
  cols[0] = sum_q(fxj, lane);
  cols[1] = sum_q(fyj, lane);
  cols[2] = sum_q(fzj, lane);
}

template <int COLS>
struct ChainRun {
  const float4* L;
  int ni, nj, lane;
  float cut2, thr2;
  int sub, nsub, h;
  float* t;
  float rows[3], cols[3];
  unsigned long long near;
  template <int CLS, bool DIAG, bool CUT, bool FULL>
  __device__ __forceinline__ void run() {
    chain_tile<CLS, DIAG, CUT, FULL, COLS>(L, ni, nj, lane, cut2, thr2, sub, nsub, h, t, rows, cols, near);
  }
};

struct ChainPass : ObcPass<ChainPass, 3> {
  template <int COLS>
  using Run = ChainRun<COLS>;
  static constexpr int kRows = 3, kScratch = kObcScratch<3>;

  __device__ __forceinline__ static float3 near_pair(const Tile4* ti, const Tile4* tj, int row, int col) {
    return chain_near_pair(ti, tj, row, col);
  }
  __device__ __forceinline__ static void add_row(float (&n)[3], const float4& c, float mine) {
    n[0] = fmaf(mine, c.x, n[0]); n[1] = fmaf(mine, c.y, n[1]); n[2] = fmaf(mine, c.z, n[2]);
  }
  __device__ __forceinline__ static void add_col(float (&m)[3], const float4& c, float mine) {
    m[0] = fmaf(-mine, c.x, m[0]); m[1] = fmaf(-mine, c.y, m[1]); m[2] = fmaf(-mine, c.z, m[2]);
  }
  __device__ __forceinline__ static void near_two(const Tile4* t, int atom, const int (&o)[2], const bool (&on)[2],
                                                  float (&even)[3], float (&odd)[3]) {
    chain_near_diag(t, atom, o, on, even, odd);
  }
  __device__ __forceinline__ static void put(const DeviceView& v, int w, int side, int at, const float (&x)[3]) {
    float* pc = part3(v, w, side);
    pc[at] = x[0];
    pc[kTile + at] = x[1];
    pc[2 * kTile + at] = x[2];
  }

  __device__ __forceinline__ bool stage(const DeviceView& v, int w_, const PairItem& it, bool rows, bool cols,
                                        float4* L) {
    w = w_;
    lane = threadIdx.x & 63;
    const SlotConst& S = v.slots[item_slot(it.meta)];
    if (skip_item(v, S, it)) return false;
    const int packed = v.item_cls[w], cls = packed & kClsMask;
    thr2 = cls_thr2(packed);
    cut = false;
    if (S.gb_cut) {
      if ((cls & kClsCutMask) == kClsFar) return false;
      cut = (cls & kClsCutMask) == kClsStraddle;
    }
    cut2 = S.cutoff2;
    lim2 = cut ? fminf(thr2, prev_below(cut2)) : thr2;
    tier = cls >> kClsTierShift;
    const JSrc js = j_source(v, it, lane);
    ItemAtoms t = load_atoms<true>(v, it, js, lane, rows, cols);
    diag = (item_flags(it.meta) & kFlagDiag) != 0;
    ni = item_ni(it.meta);
    nj = js.nj;
    full = ni == kTile && nj == kTile;
    nsub = it.nsub;
    if (!full) pad_atoms(t, lane, ni, nj);
    StageRun<ChainAtom> put{t, lane, rows, cols, L};
    by_class(tier, diag, cut, full, put);
    return true;
  }
};

// ---------------------------------------------------------------------------
// Items to waves
// ---------------------------------------------------------------------------
// The rows of an item are one share or two (PairItem.nsub, by the system's size: share s
// has the rows of patches b = s, s + nsub, ...), whose column sums are added in their
// order, and a row's sum is that of its half 0 plus that of its half 1. So one, two or
// four waves give the same sums bit for bit, in any pack and on any path:
// - a wave takes the item, its shares one after the other;
// - two waves take a share each, and the second's column sums go through LDS;
// - four waves take a half of the columns of a share each: they keep their four columns in
//   registers, and the lanes of their rows meet in LDS.
// Four row shares, whose column sums a wave alone formed four times over with four lists
// of near pairs, cost the packs 4 to 12% that a lone system gained (us a step of 303 systems
// of 700 atoms: 374, now 336; of one of 2,500: 54, now 53).
// The first two waves of an item bring its two tiles into LDS, for all. Waves of
// one, two or four items form a unit (prx_common.h).
template <class Pass>
constexpr int kWaveLds = kTilesLds + Pass::kScratch + Pass::kLaneEnergies;  // a wave's memory where it takes an item or a share
template <class Pass>
constexpr int kGroupLds =
    kUnitWaves * kWaveLds<Pass> > Pass::Quarter::kSize ? kUnitWaves * kWaveLds<Pass> : Pass::Quarter::kSize;
constexpr int kAnyWaveLds = kWaveLds<ChainPass>;                // of any pass
constexpr int kAnyGroupLds = kGroupLds<ForcePass<false>>;
static_assert(kAnyWaveLds >= kWaveLds<BornPass> && kAnyWaveLds >= kWaveLds<ForcePass<false>>, "");
static_assert(kAnyGroupLds >= kGroupLds<BornPass> && kAnyGroupLds >= kGroupLds<ChainPass> &&
                  kAnyGroupLds >= kUnitWaves * kAnyWaveLds, "");

// Wave k of a group of W takes its part of unit u; M: the group's memory. meet: the
// unit holds exactly two workgroup barriers, also one of whole items or of items
// without work (groups of one workgroup, and waves of one group, meet the same
// barriers whatever their units are); else none, and all its items are whole. LOOP:
// a wave that takes a whole item may find two shares in it. QUAD: every unit of the
// list is an item on four waves.
template <class Pass, int W, bool LOOP, bool QUAD = false>
__device__ __forceinline__ void pair_unit(const DeviceView& v, const PairUnit& u, int k, bool meet, float4* M) {
  constexpr int kWave = kWaveLds<Pass>;
  const int sh = QUAD ? kUnitWaves : u.shares;  // waves per item
  const bool four = W == kUnitWaves && sh == kUnitWaves;
  const int m = sh == W ? 0 : (sh == 1 ? k : k / 2), sub = k - m * sh;
  const int w = u.first + m;
  float4* const tiles = M + (four ? 0 : m * sh * kWave);
  float4* const own = M + k * kWave + kTilesLds;
  PairItem it;
  Pass f;
  bool on = m < u.n;
  if (on) {
    it = v.items[w];
    on = f.stage(v, w, it, sub == 0, sub == (sh > 1 ? 1 : 0), tiles);
  }
  if (meet)
    __syncthreads();
  else
    wave_lds_sync();
  typename Pass::Sum s;
  if (on) {
    if (four) {
      s = f.quarter(k, M);
    } else {
      s = f.template run<LOOP>(v, sub, sh > 1 ? sub + 1 : it.nsub, tiles, own);
      if (sub > 0) s.to_lds(own, f.lane);
    }
  }
  if (meet) __syncthreads();
  if (!on) return;
  if (four) {
    f.finish(v, k, M, s);
  } else if (sub == 0) {
    if (sh > 1) {
      typename Pass::Sum o;
      o.from_lds(own + kWave, f.lane);
      s.add(o);
    }
    f.store(v, s);
  }
}

// An item on one wave; L: the wave's memory.
template <class Pass>
__device__ __forceinline__ void pair_wave(const DeviceView& v, int w, float4* L) {
  pair_unit<Pass, 1, false>(v, PairUnit{w, 1, 1}, 0, false, L);
}

// Item or unit of block b of nb. Workgroups are dispatched to the 8 XCDs round-robin
// (block b to XCD b mod 8), and each XCD has its own L2. With PRX_XCD_MAP the
// blocks are renumbered so that XCD x runs one contiguous run of them
// (consecutive items share their i tile and neighbouring j tiles, which then
// hit in that XCD's L2, and so do the partials for the tile gathers): block
// b = 8k + x becomes x * per + min(x, rem) + k, a bijection on [0, nb) with
// per = nb / 8, rem = nb % 8. Not with neighbour lists: there most chunk items
// are empty, and more so in the first rows, so that one XCD of eight would get
// more than twice the average work (20,000 atoms cut at 20 A, Born, force, chain:
// 51, 55, 58 us; 45, 42, 50 in plain order).
constexpr int kXcds = 8;

__device__ __forceinline__ int unit_id(const DeviceView& v, int b, int nb) {
#if PRX_XCD_MAP
  if (v.nl_tp_hw > 0) return b;
  const int per = nb / kXcds, rem = nb % kXcds;
  const int x = b % kXcds, k = b / kXcds;
  b = x * per + min(x, rem) + k;
#endif
  return b;
}

// Wave of this thread within its group (wave-uniform).
template <int WAVES = kUnitWaves>
__device__ __forceinline__ int unit_wave() {
  return __builtin_amdgcn_readfirstlane((int)((threadIdx.x >> 6) & (WAVES - 1)));
}

}  // namespace prx

#pragma clang fp contract(fast)
