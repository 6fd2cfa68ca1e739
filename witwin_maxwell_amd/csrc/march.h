// Tile march: one launch advances the whole grid -- interior, CPML layers and
// faces alike -- by one or two full time steps.
//
// A block of sixteen wavefronts owns a tile of rows and columns (one z column per
// lane, one y row per wavefront) and marches along x over a chunk of planes.  Per
// plane it computes H and then E of the tile from values held in registers: the x
// neighbours are the planes before and after, the z neighbours come from the lanes
// beside (DPP shifts), the y neighbours from the wavefronts beside (LDS, two
// barriers a plane).  With T = 2 the march carries a second time step two planes
// behind the first, so E, H, the curl coefficients, the CPML psi and the running
// sums are read once and written once per TWO steps.
//
// What bounds it.  The separate interior / shell / z-end launches take a step at
// 3.3-4.0 TB/s of a 6.2 TB/s copy: they move every array once or twice per step, so the
// bytes had to go, not the latency.  Here each value loaded serves T steps; the price is
// the halo: T rows, columns and planes at each side of a tile are computed again by the
// neighbours (16 - 2T of 16 rows, 64 - 2T of 64 columns are a tile's own), whose loads
// mostly hit L2 because the blocks resident on an XCD are neighbouring tiles marching
// together.  A pass over 281^3 nodes with CPML moves 2.22 GB of HBM at 2.4 TB/s (separate
// launches 1.98 GB a step).  What is left is the rate of a CU's vector memory instructions
// (324 a wavefront of sixteen planes, 43.7 thousand a CU and pass, 51 cycles each) and the
// two barriers a plane; the wavefronts wait for half of their cycles.  us per step,
// separate launches -> march: PEC box of 257^3 370 -> 184, 129^3 47 -> 32, 65^3 19 -> 13;
// with CPML 12 and a plane wave 281^3 567 -> 424, 185^3 195 -> 174, 105^3 56 -> 45.
//
// Sixteen rows per block keep the share of halo rows low (4 of 16 at T = 2) and
// fill a CU with one block (at most 128 VGPRs), so register use up to that costs no
// occupancy: CPML, source terms and observers stay in the one kernel behind
// wave-uniform tests.
//
// Rounding.  One step taken by T = 1 and the same step inside a T = 2 march give the
// same bits (a run may be split anywhere): every update below is written with
// explicit fused multiply-adds, contraction off, and a sample's arithmetic does not
// depend on the tile it falls into.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "maxwell_fdtd.h"
#include "terms.h"
#include "yee.h"

namespace mw {

constexpr int kMarchRows = 16;   // wavefronts (rows) per block
constexpr int kMarchCols = 64;   // lanes (columns)
constexpr int kMarchPlanes = 248; // most planes a block walks
constexpr int kMarchPoints = 64; // point observers a march can take
constexpr int kMarchDft = 2;    // frequencies whose running sums are read together
constexpr int kMarchBlocks = 256; // blocks that a march lists one by one

struct MarchBlock {  // one block's tile and planes [x0, x1)
  uint16_t x0, x1;
  uint8_t y, z;
};

struct MarchPlane {  // one observed plane; its samples go to a step's stage row at `off`
  int32_t component, axis, index, off;
};

struct MarchArgs {
  mw_grid g;
  mw_coeffs cf;
  mw_cpml cp;          // psi[0..11] = input buffers
  float* psi_out[12];  // output buffers (E side: the input itself when T = 1)
  mw_fields in, out;
  // the same buffers (and the E curl coefficients) as the plane loop walks them: each
  // moved by the planes between the one the loop is at and the one it reads or writes
  const float* ahead[9];   // E two planes ahead, H and curl one plane ahead
  float* behind_e[3];      // T = 2: E two planes behind, H one plane behind; else level
  float* behind_h[3];
  const mw_term* h_terms;  // device copies of the descriptors
  const mw_term* e_terms;
  int32_t n_h_terms, n_e_terms;
  const float* line_history;  // rows of line_n floats: E^n, H^{n+1/2}, E^{n+1}, H^{n+3/2}
  int32_t line_n;
  int32_t nf_dft, n_points, n_planes, point_off;  // points: their place in a stage row
  const float* dft_cos;  // (steps, nf_dft)
  const float* dft_sin;
  float* dft_re[3];
  float* dft_im[3];
  const int32_t* point_component;
  const int32_t* point_linear;
  float* stage[2];       // the steps' stage rows of observed planes and points
  int32_t tiles_z, tiles_y, blocks;
  MarchPlane planes[MW_MAX_PLANES];
  int32_t chunk;  // > 0: every block walks so many planes, z tiles fastest, then y tiles
  MarchBlock list[kMarchBlocks];  // chunk = 0: the blocks
};

// Value of the lane below / above (0 beyond the end: the outermost lanes are halo).
// Written so that the shift folds into the subtraction that uses it.
__device__ __forceinline__ float lane_below(float v) {
#ifdef MW_EMULATED_BLOCKS
  return __shfl_up(v, 1, 64);
#else
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138 /* wave_shr:1 */,
                                                               0xf, 0xf, true));
#endif
}
__device__ __forceinline__ float lane_above(float v) {
#ifdef MW_EMULATED_BLOCKS
  return __shfl_down(v, 1, 64);
#else
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x130 /* wave_shl:1 */,
                                                               0xf, 0xf, true));
#endif
}

// Block barrier that orders LDS only: a full __syncthreads would also wait for the
// next plane's loads and the last plane's stores, which are still in flight.
__device__ __forceinline__ void lds_barrier() {
#ifdef MW_EMULATED_BLOCKS
  __syncthreads();
#else
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#endif
}

struct V3 {
  float x, y, z;
};

// Read-only view of a table that nothing in the launch writes (spacings, profiles,
// weights, descriptors): a uniform index is then read through the scalar cache
// instead of the vector memory queue, where it would wait behind the plane's loads.
template <class T>
using cptr = __attribute__((address_space(4))) const T*;
template <class T>
__device__ __forceinline__ cptr<T> C(const T* p) {
  return (cptr<T>)p;
}

// (a - b) * s, and the CPML form d / kappa + psi with psi advanced in place where
// the sample lies in the slab
__device__ __forceinline__ float slope(float a, float b, float s) {
#pragma clang fp contract(off)
  return (a - b) * s;
}
__device__ __forceinline__ float stretched(float d, float ik, float b, float c, bool in, float& psi) {
#pragma clang fp contract(off)
  const float cd = c * d;
  const float next = __builtin_fmaf(b, psi, cd);
  psi = in ? next : psi;
  return __builtin_fmaf(d, ik, in ? next : 0.0f);
}
__device__ __forceinline__ float minus(float a, float b) {
#pragma clang fp contract(off)
  return a - b;
}
__device__ __forceinline__ float scaled(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}

// The march's arguments where the launch keeps them.  `fresh`
// hides where a pointer came from, so what is read through it is read there: the
// arguments of the rarer work (layers, sums, terms) would otherwise all be hoisted
// out of the plane loop and spilled, and cost every plane of every tile.
using MarchPtr = cptr<MarchArgs>;
__device__ __forceinline__ MarchPtr fresh(MarchPtr p) {
#ifndef MW_EMULATED_BLOCKS
  uint64_t v = (uint64_t)p;
  asm volatile("" : "+s"(v));
  return (MarchPtr)v;
#else
  return p;
#endif
}

// Value of component c (0..5 = Ex..Hz) of a sample.
__device__ __forceinline__ float component_of(int c, const V3& e, const V3& h) {
  return c == 0 ? e.x : c == 1 ? e.y : c == 2 ? e.z : c == 3 ? h.x : c == 4 ? h.y : h.z;
}

// Value of term q of a family (0 H, 1 E) at sample (i, j, k) at step n + t of a march
// that starts at step n; 0 outside its patch.
__device__ __forceinline__ float march_term(MarchPtr a, int family, int q, int i, int j, int k, int n, int t) {
#pragma clang fp contract(off)
  const auto& d = C(family ? a->e_terms : a->h_terms)[q];
  const int pi = i - d.offset[0], pj = j - d.offset[1], pk = k - d.offset[2];
  if (pi < 0 || pj < 0 || pk < 0 || pi >= d.shape[0] || pj >= d.shape[1] || pk >= d.shape[2]) return 0.0f;
  const int64_t cells = (int64_t)d.shape[0] * d.shape[1] * d.shape[2];
  const int64_t p = ((int64_t)pi * d.shape[1] + pj) * d.shape[2] + pk;
  if (d.kind == MW_TERM_ADDITIVE) return C(d.signal_table)[n + t] * G(d.patch)[p];
  if (d.kind == MW_TERM_LINE) {
    const int pa = d.line_axis == 0 ? pi : (d.line_axis == 1 ? pj : pk);
    const int m = d.line_axis < 0 ? d.line_base : d.line_base + d.line_step * pa;
    return G(d.patch)[p] * G(a->line_history)[(int64_t)(2 * t + family) * a->line_n + m];
  }
  return G(d.values)[(int64_t)t * cells + p];
}

// Terms of one family that touch row j and columns [k0, k1]: the planes [lo, hi) in
// which some do, how many there are and the last of them (with its component).
struct TermReach {
  int lo, hi, count, last, component;
};
__device__ __forceinline__ TermReach term_reach(const mw_term* __restrict__ t, int n, int j, int k0, int k1) {
  TermReach r{1 << 30, 0, 0, 0, 0};
  for (int q = 0; q < n; ++q) {
    const auto& d = C(t)[q];
    if (j >= d.offset[1] && j < d.offset[1] + d.shape[1] && k1 >= d.offset[2] && k0 < d.offset[2] + d.shape[2]) {
      r.lo = min(r.lo, (int)d.offset[0]);
      r.hi = max(r.hi, (int)(d.offset[0] + d.shape[0]));
      r.count += 1;
      r.last = q;
      r.component = d.component;
    }
  }
  return r;
}

// Face rule of one E sample along one axis: 0 inside, else the boundary mode with
// the end it sits at.
struct Face {
  bool pec, held, pmc_lo, pmc_hi;  // held: PEC or left as it is (no boundary, CPML)
};
__device__ __forceinline__ Face face_rule(int x, int n, int lo, int hi) {
  Face f;
  f.pec = face_pec(x, n, lo, hi);
  f.held = f.pec || face_inactive(x, n, lo, hi);
  f.pmc_lo = x == 0 && lo == MW_BC_PMC;
  f.pmc_hi = x + 1 == n && hi == MW_BC_PMC;
  return f;
}
// derivative at a face sample: the PMC mirror where that is the rule
__device__ __forceinline__ float mirrored(float d, const Face& f, float cur, float prev, float inv) {
#pragma clang fp contract(off)
  if (f.pmc_lo) return 2.0f * cur * inv;
  if (f.pmc_hi) return -2.0f * prev * inv;
  return d;
}

// The one shifted or additive term of a family (H, E) that a row meets, as the row
// reads it: the row's first sample in the term's first plane (null: none, or a line
// term), the samples from plane to plane and from step to step, the steps' factors,
// and the columns it covers.
struct MarchSheet {
  const float* row;
  uint32_t plane, next;
  float scale[2];
  int32_t first, columns;
};

// LDS of a block: the row exchanges (x and z components of E^n, H^{n+1/2} and, at
// T = 2, E^{n+1}, H^{n+3/2}) and the decoded point observers.
template <int T>
struct MarchShared {
  float e1x[kMarchRows][kMarchCols], e1z[kMarchRows][kMarchCols];
  float h1x[kMarchRows][kMarchCols], h1z[kMarchRows][kMarchCols];
  float e2x[T == 2 ? kMarchRows : 1][kMarchCols], e2z[T == 2 ? kMarchRows : 1][kMarchCols];
  float h2x[T == 2 ? kMarchRows : 1][kMarchCols], h2z[T == 2 ? kMarchRows : 1][kMarchCols];
  int pi[kMarchPoints], pj[kMarchPoints], pk[kMarchPoints], pc[kMarchPoints];
  float ihx[kMarchPlanes + 8], iex[kMarchPlanes + 8];  // x spacings of the march's planes
  float yp[6][kMarchRows], zp[6][kMarchCols];  // CPML profiles of the rows / lanes: 1/kappa, b, c of H, then E
  // observed planes.  z planes, of which a row meets one sample: their slot by
  // component and lane (< 0: none) and the last samples by step, slot and row, which
  // a few wavefronts then store for the whole block (a store costs as much for one
  // lane as for 64).  The first place of each row in a y plane, by component, and the
  // x planes (a mask of the descriptors) at each plane of the march.
  int slot_z[6][kMarchCols], place_y[6][kMarchRows];
  float sample_z[2][MW_MAX_PLANES][kMarchRows];
  uint32_t planes_x[kMarchPlanes + 8];
  MarchSheet sheets[2][kMarchRows];
  // T = 2: each thread's CPML psi after the first step, by plane parity, until the
  // second step of that plane (24 values a thread would not fit the registers)
  float qh[T == 2 ? 12 : 1][kMarchRows][kMarchCols], qe[T == 2 ? 12 : 1][kMarchRows][kMarchCols];
};

// Sample of a plane's row: `row` is uniform over the wavefront, the lane adds a byte
// offset.  The row's address is pinned to scalar registers: left alone, loop strength
// reduction turns every array's address into a 64-bit vector induction variable, and
// thirty of those do not fit beside the march.
template <class T>
__device__ __forceinline__ gptr<T> pinned(T* row) {
  uint64_t p = (uint64_t)row;
#ifndef MW_EMULATED_BLOCKS
  p = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)p) |
      (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(p >> 32)) << 32;
  asm("" : "+s"(p));
#endif
  return (gptr<T>)p;
}
__device__ __forceinline__ float row_load(const float* row, uint32_t lane_bytes) {
  return *(gptr<const float>)((gptr<const char>)pinned(row) + lane_bytes);
}
__device__ __forceinline__ void row_store(float* row, uint32_t lane_bytes, float v) {
  *(gptr<float>)((gptr<char>)pinned(row) + lane_bytes) = v;
}
// Waits for every load and store issued so far.  Loads and stores retire in order
// through one counter, and behind stores that a plane may or may not make the
// compiler cannot count: without this one wait, placed after a plane's loads have had
// half the plane's work to arrive and before its first store, it drains the counter
// again and again.
__device__ __forceinline__ void memory_settled() {
#ifndef MW_EMULATED_BLOCKS
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0); the other counters untouched
#endif
}

// A uniform integer held in a scalar register (and known to be uniform, wherever the
// compiler found it); a uniform float held in a vector register, of which the march
// has more to spare.
__device__ __forceinline__ int held(int x) {
#ifndef MW_EMULATED_BLOCKS
  x = __builtin_amdgcn_readfirstlane(x);
  asm volatile("" : "+s"(x));
#endif
  return x;
}
template <class T>
__device__ __forceinline__ T* uniform(T* x) {
  const uint64_t p = (uint64_t)x;
#ifndef MW_EMULATED_BLOCKS
  return (T*)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)p) |
              (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(p >> 32)) << 32);
#else
  return (T*)p;
#endif
}
__device__ __forceinline__ float spread(float x) {
#ifndef MW_EMULATED_BLOCKS
  asm("" : "+v"(x));
#endif
  return x;
}

// Six consecutive addresses from the arguments, all fetched here.
template <class P, class T>
__device__ __forceinline__ void fetched(P from, T** to) {
#pragma unroll
  for (int q = 0; q < 6; ++q) to[q] = (T*)from[q];
#ifndef MW_EMULATED_BLOCKS
  asm volatile("" : "+s"(to[0]), "+s"(to[1]), "+s"(to[2]), "+s"(to[3]), "+s"(to[4]), "+s"(to[5]));
#endif
}

// What a wavefront meets on its march (uniform).
enum : uint32_t {
  kLayerHy = 1, kLayerEy = 2, kLayerHz = 4, kLayerEz = 8,  // CPML layers of its row / of some lane
  kLayerX = 16,                                            // CPML layers of some plane
  kLayers = 31,
  kFaceYZ = 32,    // its row or some lane on a y or z face
  kWatch = 64,     // an observer of its own samples
  kHeldY = 256, kPecY = 512,  // its row on a held / PEC y face
  kMirror = 1024,             // the grid has a PMC face
};

// COEF: coefficient mode of the scene (fused.h): 0 general, 1 E curl arrays only,
// 2 uniform.  DFT: with the full-field running sums (in kernels of their own: beside
// them the others lost 7-10 % to spilled scalars).  `logical` = number of the block.
template <int T, int COEF, bool DFT>
__device__ __forceinline__ void march_block(MarchPtr a, int n, int logical, MarchShared<T>& sh) {
  const int nx = held(a->g.nx), ny = held(a->g.ny), nz = held(a->g.nz);
  const int tiles_z = a->tiles_z, tiles_y = a->tiles_y;
  int tz, ty, i0, i1;
  if (a->chunk > 0) {
    tz = logical % tiles_z;
    ty = (logical / tiles_z) % tiles_y;
    i0 = logical / (tiles_z * tiles_y) * a->chunk;
    i1 = min(i0 + a->chunk, nx);
  } else {
    const auto& of = a->list[logical];
    tz = of.z;
    ty = of.y;
    i0 = of.x0;
    i1 = of.x1;
  }
  tz = held(tz), ty = held(ty), i0 = held(i0), i1 = held(i1);
  const int lane = threadIdx.x, row = wave_row();
  const int up = min(row + 1, kMarchRows - 1), down = max(row - 1, 0);
  const int k0 = tz * (kMarchCols - 2 * T), k = k0 + lane;
  const int j = ty * (kMarchRows - 2 * T) + row;
  const int p0 = max(i0 - T, 0);
  const int first_last = min(T == 2 ? i1 : i1 - 1, nx - 1);  // last plane of the first step
  const int p1 = T == 2 ? i1 + 1 : i1 - 1;
  const int nx1 = held(nx - 1), nx2 = held(nx - 2);
  const int steady = held(nx - 4);  // up to this plane every component has the planes ahead
  // the samples this thread's tile owns: all but T rows and columns at each inner
  // side of the tile (`n`: components with a sample on every node of the axis, `m`:
  // with one fewer)
  const bool own_k = (tz == 0 || lane >= T) && (tz == tiles_z - 1 || lane < kMarchCols - T);
  const bool own_j = (ty == 0 || row >= T) && (ty == tiles_y - 1 || row < kMarchRows - T);
  const bool kn_ok = own_k && k < nz, km_ok = own_k && k < nz - 1;
  const bool jn_ok = own_j && j < ny, jm_ok = own_j && j < ny - 1;
  // coordinates that exist, for the addresses of lanes and rows beyond the grid
  const int kn = min(k, nz - 1), km = min(k, nz - 2), jn = min(j, ny - 1), jm = min(j, ny - 2);
  const uint32_t kn4 = 4u * (uint32_t)kn, km4 = 4u * (uint32_t)km;
  // plane sizes by (rows, columns), and a row's place in its plane
  const uint32_t snn = (uint32_t)ny * nz, smn = (uint32_t)(ny - 1) * nz, snm = (uint32_t)ny * (nz - 1),
                 smm = (uint32_t)(ny - 1) * (nz - 1);
  const uint32_t rnn = (uint32_t)jn * nz, rmn = (uint32_t)jm * nz, rnm = (uint32_t)jn * (nz - 1),
                 rmm = (uint32_t)jm * (nz - 1);
  auto pn = [&](int i) { return (uint32_t)min(i, nx1); };  // plane of Ey, Ez, Hx
  auto pm = [&](int i) { return (uint32_t)min(i, nx2); };  // plane of Ex, Hy, Hz
  const float ihz = C(a->g.inv_h[2])[km], iez = C(a->g.inv_e[2])[kn];
  const float ihy = spread(C(a->g.inv_h[1])[jm]), iey = spread(C(a->g.inv_e[1])[jn]);

  // CPML layers (outside them kappa = 1 and c = 0, so only samples inside matter); the
  // profiles wait in LDS for the wavefronts that meet a layer
  uint32_t met = 0;
  int lyh = -1, lye = -1, lzh = -1, lze = -1;
  auto slab = [](MarchPtr f, int q, int x) {
    return slab_local(x, f->cp.psi_low[q], f->cp.psi_high_start[q], f->cp.psi_high_len[q]);
  };
  if (a->cp.enabled) {
    lyh = j < ny - 1 ? slab(a, 6, j) : -1;
    lye = j < ny ? slab(a, 0, j) : -1;
    lzh = k < nz - 1 ? slab(a, 7, k) : -1;
    lze = k < nz ? slab(a, 1, k) : -1;
    if (lane == 0 && lyh >= 0) {
      sh.yp[0][row] = C(a->cp.inv_kappa_h[1])[j]; sh.yp[1][row] = C(a->cp.b_h[1])[j]; sh.yp[2][row] = C(a->cp.c_h[1])[j];
    }
    if (lane == 0 && lye >= 0) {
      sh.yp[3][row] = C(a->cp.inv_kappa_e[1])[j]; sh.yp[4][row] = C(a->cp.b_e[1])[j]; sh.yp[5][row] = C(a->cp.c_e[1])[j];
    }
    if (row == 0) {
      const bool h = lzh >= 0, e = lze >= 0;
      sh.zp[0][lane] = h ? C(a->cp.inv_kappa_h[2])[k] : 1.0f;
      sh.zp[1][lane] = h ? C(a->cp.b_h[2])[k] : 0.0f;
      sh.zp[2][lane] = h ? C(a->cp.c_h[2])[k] : 0.0f;
      sh.zp[3][lane] = e ? C(a->cp.inv_kappa_e[2])[k] : 1.0f;
      sh.zp[4][lane] = e ? C(a->cp.b_e[2])[k] : 0.0f;
      sh.zp[5][lane] = e ? C(a->cp.c_e[2])[k] : 0.0f;
    }
    if (lyh >= 0) met |= kLayerHy;
    if (lye >= 0) met |= kLayerEy;
    if (__ballot(lzh >= 0) != 0) met |= kLayerHz;
    if (__ballot(lze >= 0) != 0) met |= kLayerEz;
    if (p0 < max(a->cp.psi_low[8], a->cp.psi_low[2]) || (a->cp.psi_high_len[8] > 0 && p1 >= a->cp.psi_high_start[8]) ||
        (a->cp.psi_high_len[2] > 0 && p1 >= a->cp.psi_high_start[2]))
      met |= kLayerX;
  }
  if (j == 0 || j >= ny - 1 || k0 == 0 || k0 + kMarchCols >= nz) met |= kFaceYZ;
  const Face face_y = face_rule(j, ny, a->g.bc_lo[1], a->g.bc_hi[1]);
  const Face face_z = face_rule(k, nz, a->g.bc_lo[2], a->g.bc_hi[2]);
  const int face_k = (face_z.held ? 1 : 0) + (face_z.pec ? 2 : 0);
  if (face_y.held) met |= kHeldY;
  if (face_y.pec) met |= kPecY;
#pragma unroll
  for (int q = 0; q < 3; ++q)
    if (a->g.bc_lo[q] == MW_BC_PMC || a->g.bc_hi[q] == MW_BC_PMC) met |= kMirror;
  const uint32_t zh4 = 4u * (uint32_t)max(lzh, 0), ze4 = 4u * (uint32_t)max(lze, 0);

  // Source terms.  Where one term of a family meets this wavefront (a plane-wave sheet
  // crosses a wavefront in every plane), its samples are read a plane ahead; where
  // several do, when they are added.
  const TermReach ht = term_reach(a->h_terms, a->n_h_terms, j, k0, k0 + kMarchCols - 1);
  const TermReach et = term_reach(a->e_terms, a->n_e_terms, j, k0, k0 + kMarchCols - 1);
  float tv[2][2] = {{0, 0}, {0, 0}}, tv_l[2][2] = {{0, 0}, {0, 0}};  // [family][step]: samples of this plane's updates, of the next one's
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const TermReach& r = f ? et : ht;
    MarchSheet s{nullptr, 0u, 0u, {1.0f, 1.0f}, 0, 0};
    if (r.count == 1) {
      const auto& d = C(f ? a->e_terms : a->h_terms)[r.last];
      if (d.kind != MW_TERM_LINE) {
        s.plane = (uint32_t)d.shape[1] * (uint32_t)d.shape[2];
        s.row = (d.kind == MW_TERM_ADDITIVE ? d.patch : d.values) + (uint64_t)(uint32_t)(j - d.offset[1]) * (uint32_t)d.shape[2];
        s.first = d.offset[2];
        s.columns = d.shape[2];
        if (d.kind == MW_TERM_ADDITIVE) {
          for (int t = 0; t < T; ++t) s.scale[t] = C(d.signal_table)[n + t];
        } else {
          s.next = s.plane * (uint32_t)d.shape[0];
        }
      }
    }
    if (lane == 0) sh.sheets[f][row] = s;
  }
  // the samples of planes i0, i1 that the two steps add
  auto sheet = [&](int family, int i0, int i1, float* v) {
    const TermReach& r = family ? et : ht;
    if (i0 < r.lo || i1 >= r.hi) return;  // i1 <= i0
    const MarchSheet s = sh.sheets[family][row];
    const float* base = uniform(s.row);
    if (base == nullptr) {
      if (i0 >= r.lo && i0 < r.hi) v[0] = march_term(fresh(a), family, r.last, i0, j, k, n, 0);
      if (T == 2 && i1 >= r.lo && i1 < r.hi) v[1] = march_term(fresh(a), family, r.last, i1, j, k, n, 1);
      return;
    }
    const uint32_t plane = (uint32_t)held((int)s.plane), next = (uint32_t)held((int)s.next);
    const uint32_t at = (uint32_t)(k - s.first);
    if (at >= (uint32_t)s.columns) return;
    if (i0 >= r.lo && i0 < r.hi) v[0] = s.scale[0] * row_load(base + (uint64_t)(uint32_t)(i0 - r.lo) * plane, 4u * at);
    if (T == 2 && i1 >= r.lo && i1 < r.hi)
      v[1] = s.scale[1] * row_load(base + ((uint64_t)(uint32_t)(i1 - r.lo) * plane + next), 4u * at);
  };
  auto add_terms = [&](int family, int i, int t, V3& v) {
#pragma clang fp contract(off)
    const TermReach& r = family ? et : ht;
    if (i < r.lo || i >= r.hi) return;
    const int base = family ? 0 : 3;
    if (r.count == 1) {
      const float s = tv[family][t];
      if (r.component == base) v.x = v.x + s;
      else if (r.component == base + 1) v.y = v.y + s;
      else v.z = v.z + s;
      return;
    }
    const MarchPtr f = fresh(a);
    V3 sum{0.0f, 0.0f, 0.0f};
    for (int q = 0; q < (family ? f->n_e_terms : f->n_h_terms); ++q) {
      const int c = C(family ? f->e_terms : f->h_terms)[q].component - base;
      const float s = march_term(f, family, q, i, j, k, n, t);
      if (c == 0) sum.x = sum.x + s;
      else if (c == 1) sum.y = sum.y + s;
      else sum.z = sum.z + s;
    }
    v.x = v.x + sum.x;
    v.y = v.y + sum.y;
    v.z = v.z + sum.z;
  };

  // observed planes met by this wavefront's own samples: masks of the components that
  // a z plane or this row's y plane takes
  uint32_t watch_z = 0u, watch_y = 0u, watch_x = 0u;
  int slots = 0;                     // z planes of the block
  int z_place = -1, z_rows = 0, z_planes = 0;  // this lane's (slot, row) of the samples it stores, its strides
  auto rows_m = [](int c) { return c == 1 || c == 3 || c == 5; };  // one row fewer than nodes
  auto cols_m = [](int c) { return c == 2 || c == 3 || c == 4; };
  auto planes_m = [](int c) { return c == 0 || c > 3; };
  const bool z_stores = row < (MW_MAX_PLANES * kMarchRows) / kMarchCols;
  for (int q = 0; q < a->n_planes; ++q) {
    const auto& o = a->planes[q];
    const int c = o.component;
    if (o.axis == 2) {
      if (o.index < k0 + (tz == 0 ? 0 : T) || (tz < tiles_z - 1 && o.index >= k0 + kMarchCols - T)) continue;
      if (row == 0 && ((watch_z >> c & 1u) == 0u || o.index == k)) sh.slot_z[c][lane] = o.index == k ? slots : -1;
      watch_z |= 1u << c;
      if (z_stores && slots == 4 * row + lane / kMarchRows) {
        const int r = lane % kMarchRows, jr = ty * (kMarchRows - 2 * T) + r;
        const bool mine = (ty == 0 || r >= T) && (ty == tiles_y - 1 || r < kMarchRows - T) && jr < (rows_m(c) ? ny - 1 : ny);
        z_place = mine ? o.off + jr : -1;
        z_rows = rows_m(c) ? ny - 1 : ny;
        z_planes = planes_m(c) ? nx - 1 : nx;
      }
      ++slots;
      continue;
    }
    const bool mine = (rows_m(c) ? jm_ok : jn_ok) && (cols_m(c) ? km_ok : kn_ok);
    const bool hit = __ballot(mine) != 0 && (o.axis == 0 ? o.index >= i0 && o.index < i1 : o.index == j);
    if (!hit) continue;
    if (o.axis == 1) {
      sh.place_y[c][row] = o.off;
      watch_y |= 1u << c;
    } else {
      watch_x |= 1u << q;
    }
  }
  uint64_t point_mask = 0;
  if (a->n_points > 0) {
    const int points = a->n_points;
    if (row == 0 && lane < points) {
      const int c = C(a->point_component)[lane];
      const uint32_t lin = C(a->point_linear)[lane];
      const uint32_t sy = (c == 1 || c == 3 || c == 5) ? ny - 1 : ny, sz = (c == 2 || c == 3 || c == 4) ? nz - 1 : nz;
      sh.pc[lane] = c;
      sh.pk[lane] = lin % sz;
      sh.pj[lane] = (lin / sz) % sy;
      sh.pi[lane] = lin / (sz * sy);
    }
    lds_barrier();
    const bool hit = lane < points && own_j && sh.pj[lane] == j && sh.pi[lane] >= i0 && sh.pi[lane] < i1 &&
                     sh.pk[lane] >= k0 + (tz == 0 ? 0 : T) &&
                     (tz == tiles_z - 1 || sh.pk[lane] < k0 + kMarchCols - T);
    point_mask = __ballot(hit);
  }
  if ((watch_z | watch_y | watch_x) != 0u || point_mask != 0) met |= kWatch;
  // the plane loop reads this copy afresh for each plane: its tests would otherwise
  // be made once and their results kept (and spilled) as lane masks
  uint32_t flags = met;

  // samples of plane i at step n + t
  auto observe = [&](int t, int i, const V3& e, const V3& h) {
    const MarchPtr f = fresh(a);
    if ((watch_z | watch_y | watch_x) != 0u) {
      float* stage = f->stage[t];
#pragma unroll
      for (int c = 0; c < 6; ++c)
        if (((watch_z | watch_y) >> c & 1u) != 0u && i < (planes_m(c) ? nx - 1 : nx)) {
          if ((watch_z >> c & 1u) != 0u) {
            const int at = sh.slot_z[c][lane];
            if (at >= 0) sh.sample_z[t][at][row] = component_of(c, e, h);
          }
          if ((watch_y >> c & 1u) != 0u && jn_ok && (cols_m(c) ? km_ok : kn_ok))
            row_store(stage + ((int64_t)i * (cols_m(c) ? nz - 1 : nz) + held(sh.place_y[c][row])), 4u * (uint32_t)k,
                      component_of(c, e, h));
        }
      if (watch_x != 0u)
        for (uint32_t m = (uint32_t)held((int)(watch_x & sh.planes_x[i - p0])); m != 0u; m &= m - 1u) {
          const auto& o = f->planes[__builtin_ctz(m)];
          const int c = o.component;
          if ((rows_m(c) ? jm_ok : jn_ok) && (cols_m(c) ? km_ok : kn_ok))
            row_store(stage + ((int64_t)o.off + (int64_t)j * (cols_m(c) ? nz - 1 : nz)), 4u * (uint32_t)k,
                      component_of(c, e, h));
        }
    }
    for (uint64_t m = point_mask; m != 0; m &= m - 1) {
      const int q = __builtin_ctzll(m);
      if (sh.pi[q] != i || sh.pk[q] != k) continue;
      const int c = sh.pc[q];
      f->stage[t][f->point_off + q] = component_of(c, e, h);
    }
  };

  // the z planes' samples of iteration p, a barrier later: step n's of plane p and, at
  // T = 2, step n + 1's of plane p - 2
  auto store_z = [&](int p) {
    if (!z_stores || 4 * row >= slots) return;
    const MarchPtr f = fresh(a);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int i = t ? p - 2 : p;
      if (i < i0 || i >= i1) continue;
      if (z_place >= 0 && i < z_planes)
        row_store(f->stage[t], 4u * (uint32_t)(z_place + i * z_rows), sh.sample_z[t][4 * row + lane / kMarchRows][lane % kMarchRows]);
    }
  };

  // H of plane i from E of that plane (`e`, with its row and lane neighbours), the
  // next plane's E and the old H; `psi` = the six H-side psi values (hx_y hx_z hy_x
  // hy_z hz_x hz_y), advanced
  const float nhx = spread(-a->cf.curl_value[3]), nhy = spread(-a->cf.curl_value[4]), nhz = spread(-a->cf.curl_value[5]);
  auto update_h = [&](int i, int t, float ihx, const V3& e, float ex_j, float ez_j, const V3& en, const V3& old,
                      float* psi) {
    const float ex_k = lane_above(e.x), ey_k = lane_above(e.y);
    // y derivatives (and yx) as a difference and its factor, which the curl's fused
    // multiply-add takes together; a stretched one is whole, with factor 1
    float xy = minus(ez_j, e.z), xz = slope(ey_k, e.y, ihz);
    float yx = minus(en.z, e.z), yz = slope(ex_k, e.x, ihz);
    float zx = slope(en.y, e.y, ihx), zy = minus(ex_j, e.x);
    float wy = ihy, wx = ihx;
    if (flags & (kLayerHy | kLayerHz | kLayerX)) {
      if (flags & kLayerHy) {
        const float ik = sh.yp[0][row], b = sh.yp[1][row], c = sh.yp[2][row];
        xy = stretched(scaled(xy, ihy), ik, b, c, true, psi[0]);
        zy = stretched(scaled(zy, ihy), ik, b, c, true, psi[5]);
        wy = 1.0f;
      }
      if (flags & kLayerHz) {
        const float ik = sh.zp[0][lane], b = sh.zp[1][lane], c = sh.zp[2][lane];
        xz = stretched(xz, ik, b, c, lzh >= 0, psi[1]);
        yz = stretched(yz, ik, b, c, lzh >= 0, psi[3]);
      }
      if ((flags & kLayerX) && i < nx - 1) {
        const MarchPtr f = fresh(a);
        if (slab(f, 8, i) >= 0) {
          const float ik = C(f->cp.inv_kappa_h[0])[i], b = C(f->cp.b_h[0])[i], c = C(f->cp.c_h[0])[i];
          yx = stretched(scaled(yx, ihx), ik, b, c, true, psi[2]);
          wx = 1.0f;
          zx = stretched(zx, ik, b, c, true, psi[4]);
        }
      }
    }
    const float cx = __builtin_fmaf(xy, wy, -xz), cy = __builtin_fmaf(-yx, wx, yz), cz = __builtin_fmaf(-zy, wy, zx);
    V3 h;
    if (COEF == 0) {
      const MarchPtr f = fresh(a);
      auto value = [&](const float* arr, float scalar, uint64_t first, uint32_t lane4) {
        return arr ? row_load(arr + first, lane4) : scalar;
      };
      const uint32_t ox = pn(i) * smm + rmm, oy = pm(i) * snm + rnm, oz = pm(i) * smn + rmn;
      h.x = __builtin_fmaf(old.x, value(f->cf.decay[3], f->cf.decay_value[3], ox, km4), -scaled(value(f->cf.curl[3], f->cf.curl_value[3], ox, km4), cx));
      h.y = __builtin_fmaf(old.y, value(f->cf.decay[4], f->cf.decay_value[4], oy, km4), -scaled(value(f->cf.curl[4], f->cf.curl_value[4], oy, km4), cy));
      h.z = __builtin_fmaf(old.z, value(f->cf.decay[5], f->cf.decay_value[5], oz, kn4), -scaled(value(f->cf.curl[5], f->cf.curl_value[5], oz, kn4), cz));
    } else {
      h.x = __builtin_fmaf(nhx, cx, old.x);
      h.y = __builtin_fmaf(nhy, cy, old.y);
      h.z = __builtin_fmaf(nhz, cz, old.z);
    }
    add_terms(0, i, t, h);
    return h;
  };

  // E of plane i from H of that plane (`h`, with its row and lane neighbours) and of
  // the plane before, the old E and the E coefficients (`kc` curl, `kd` decay; psi
  // order ex_y ex_z ey_x ey_z ez_x ez_y)
  auto update_e = [&](int i, int t, float iex, const V3& h, float hx_j, float hz_j, float hy_i, float hz_i,
                      const V3& old, const V3& kc, const V3& kd, float* psi) {
    const float hx_k = lane_below(h.x), hy_k = lane_below(h.y);
    float xy = minus(h.z, hz_j), xz = slope(h.y, hy_k, iez);
    float yx = minus(h.z, hz_i), yz = slope(h.x, hx_k, iez);
    float zx = slope(h.y, hy_i, iex), zy = minus(h.x, hx_j);
    float wy = iey, wx = iex;
    bool held_x = false, held_y = false, held_z = false, pec_x = false, pec_y = false, pec_z = false;
    const bool faces = (flags & kFaceYZ) != 0 || i == 0 || i == nx - 1;
    if (faces) {
      const MarchPtr f = fresh(a);
      const Face fx = face_rule(i, nx, f->g.bc_lo[0], f->g.bc_hi[0]);
      if (flags & kMirror) {
        const Face fy = face_rule(j, ny, f->g.bc_lo[1], f->g.bc_hi[1]);
        const Face fz = face_rule(k, nz, f->g.bc_lo[2], f->g.bc_hi[2]);
        xz = mirrored(xz, fz, h.y, hy_k, iez);
        yz = mirrored(yz, fz, h.x, hx_k, iez);
        zx = mirrored(zx, fx, h.y, hy_i, iex);
        if (fy.pmc_lo || fy.pmc_hi) {
          xy = mirrored(xy, fy, h.z, hz_j, iey);
          zy = mirrored(zy, fy, h.x, hx_j, iey);
          wy = 1.0f;
        }
        if (fx.pmc_lo || fx.pmc_hi) {
          yx = mirrored(yx, fx, h.z, hz_i, iex);
          wx = 1.0f;
        }
      }
      const bool held_j = (flags & kHeldY) != 0, pec_j = (flags & kPecY) != 0, held_k = (face_k & 1) != 0,
                 pec_k = (face_k & 2) != 0;
      held_x = held_j || held_k; pec_x = pec_j || pec_k;
      held_y = fx.held || held_k; pec_y = fx.pec || pec_k;
      held_z = fx.held || held_j; pec_z = fx.pec || pec_j;
    }
    if (flags & (kLayerEy | kLayerEz | kLayerX)) {  // the psi of a sample held by its face stays as it is
      if (flags & kLayerEy) {
        const float ik = sh.yp[3][row], b = sh.yp[4][row], c = sh.yp[5][row];
        xy = stretched(scaled(xy, wy), ik, b, c, !held_x, psi[0]);
        zy = stretched(scaled(zy, wy), ik, b, c, !held_z, psi[5]);
        wy = 1.0f;
      }
      if (flags & kLayerEz) {
        const float ik = sh.zp[3][lane], b = sh.zp[4][lane], c = sh.zp[5][lane];
        xz = stretched(xz, ik, b, c, lze >= 0 && !held_x, psi[1]);
        yz = stretched(yz, ik, b, c, lze >= 0 && !held_y, psi[3]);
      }
      if ((flags & kLayerX) && i < nx) {
        const MarchPtr f = fresh(a);
        if (slab(f, 2, i) >= 0) {
          const float ik = C(f->cp.inv_kappa_e[0])[i], b = C(f->cp.b_e[0])[i], c = C(f->cp.c_e[0])[i];
          yx = stretched(scaled(yx, wx), ik, b, c, !held_y, psi[2]);
          wx = 1.0f;
          zx = stretched(zx, ik, b, c, !held_z, psi[4]);
        }
      }
    }
    const float cx = __builtin_fmaf(xy, wy, -xz), cy = __builtin_fmaf(-yx, wx, yz), cz = __builtin_fmaf(-zy, wy, zx);
    V3 e, gain = kc;
    if (COEF == 0) {
      e.x = __builtin_fmaf(old.x, kd.x, scaled(gain.x, cx));
      e.y = __builtin_fmaf(old.y, kd.y, scaled(gain.y, cy));
      e.z = __builtin_fmaf(old.z, kd.z, scaled(gain.z, cz));
    } else {
      e.x = __builtin_fmaf(gain.x, cx, old.x);
      e.y = __builtin_fmaf(gain.y, cy, old.y);
      e.z = __builtin_fmaf(gain.z, cz, old.z);
    }
    if (faces) {
      e.x = held_x ? old.x : e.x;
      e.y = held_y ? old.y : e.y;
      e.z = held_z ? old.z : e.z;
    }
    add_terms(1, i, t, e);
    if (faces) {
      e.x = pec_x ? 0.0f : e.x;
      e.y = pec_y ? 0.0f : e.y;
      e.z = pec_z ? 0.0f : e.z;
    }
    return e;
  };

  // E coefficients of plane i where the scene has arrays (COEF 0; COEF 1 moves its
  // rows along with the fields')
  const V3 curl_value{a->cf.curl_value[0], a->cf.curl_value[1], a->cf.curl_value[2]};
  auto load_general = [&](const float* x, const float* y, const float* z, V3 v, int i) {
    if (x) v.x = row_load(x + (pm(i) * snn + rnn), kn4);
    if (y) v.y = row_load(y + (pn(i) * smn + rmn), kn4);
    if (z) v.z = row_load(z + (pn(i) * snm + rnm), km4);
    return v;
  };
  auto load_curl = [&](int i) {
    const MarchPtr f = fresh(a);
    return load_general(f->cf.curl[0], f->cf.curl[1], f->cf.curl[2], curl_value, i);
  };
  auto load_decay = [&](int i) {
    const MarchPtr f = fresh(a);
    return load_general(f->cf.decay[0], f->cf.decay[1], f->cf.decay[2],
                        V3{f->cf.decay_value[0], f->cf.decay_value[1], f->cf.decay_value[2]}, i);
  };
  // the psi samples of plane i: `op(slot, first sample of the row, lane offset, whether
  // this thread owns it)` for the layers this wavefront meets.  The arrays' addresses
  // are fetched together, ahead of the tests: one wait, not one per layer.
  const uint32_t len_hy = a->cp.psi_low[6] + a->cp.psi_high_len[6], len_hz = a->cp.psi_low[7] + a->cp.psi_high_len[7],
                 len_ey = a->cp.psi_low[0] + a->cp.psi_high_len[0], len_ez = a->cp.psi_low[1] + a->cp.psi_high_len[1];
  auto each_psi_h = [&](int i, auto&& op) {
    const bool im = i < nx - 1;
    if (flags & kLayerHy) {
      op(0, (uint64_t)(pn(i) * len_hy + lyh) * (nz - 1), km4, jm_ok && km_ok);
      op(5, (uint64_t)(pm(i) * len_hy + lyh) * nz, kn4, im && jm_ok && kn_ok);
    }
    if (flags & kLayerHz) {
      op(1, (uint64_t)(pn(i) * (ny - 1) + jm) * len_hz, zh4, lzh >= 0 && jm_ok && km_ok);
      op(3, (uint64_t)(pm(i) * ny + jn) * len_hz, zh4, lzh >= 0 && im && jn_ok && km_ok);
    }
    const int l = (flags & kLayerX) && im ? slab(fresh(a), 8, i) : -1;
    if (l >= 0) {
      op(2, (uint64_t)((uint32_t)l * ny + jn) * (nz - 1), km4, jn_ok && km_ok);
      op(4, (uint64_t)((uint32_t)l * (ny - 1) + jm) * nz, kn4, jm_ok && kn_ok);
    }
  };
  auto each_psi_e = [&](int i, auto&& op) {
    const bool im = i < nx - 1;
    if (flags & kLayerEy) {
      op(0, (uint64_t)(pm(i) * len_ey + lye) * nz, kn4, im && jn_ok && kn_ok);
      op(5, (uint64_t)(pn(i) * len_ey + lye) * (nz - 1), km4, jn_ok && km_ok);
    }
    if (flags & kLayerEz) {
      op(1, (uint64_t)(pm(i) * ny + jn) * len_ez, ze4, lze >= 0 && im && jn_ok && kn_ok);
      op(3, (uint64_t)(pn(i) * (ny - 1) + jm) * len_ez, ze4, lze >= 0 && jm_ok && kn_ok);
    }
    const int l = (flags & kLayerX) && i < nx ? slab(fresh(a), 2, i) : -1;
    if (l >= 0) {
      op(2, (uint64_t)((uint32_t)l * (ny - 1) + jm) * nz, kn4, jm_ok && kn_ok);
      op(4, (uint64_t)((uint32_t)l * ny + jn) * (nz - 1), km4, jn_ok && km_ok);
    }
  };
  auto load_psi = [&](int i, float* h, float* e) {
    const MarchPtr f = fresh(a);
    const float* q[12];
    fetched(&f->cp.psi[0], q);
    fetched(&f->cp.psi[6], q + 6);
    each_psi_h(i, [&](int s, uint64_t first, uint32_t l4, bool) { h[s] = row_load(q[6 + s] + first, l4); });
    each_psi_e(i, [&](int s, uint64_t first, uint32_t l4, bool) { e[s] = row_load(q[s] + first, l4); });
  };
  auto store_psi_h = [&](int i, const float* psi) {
    float* q[6];
    fetched(&fresh(a)->psi_out[6], q);
    each_psi_h(i, [&](int s, uint64_t first, uint32_t l4, bool own) {
      if (own) row_store(q[s] + first, l4, psi[s]);
    });
  };
  auto store_psi_e = [&](int i, const float* psi) {
    float* q[6];
    fetched(&fresh(a)->psi_out[0], q);
    each_psi_e(i, [&](int s, uint64_t first, uint32_t l4, bool own) {
      if (own) row_store(q[s] + first, l4, psi[s]);
    });
  };
  // this thread's psi values of a plane to and from LDS (the axes with layers only)
  auto keep_psi = [&](float (*slot)[kMarchRows][kMarchCols], uint32_t y, uint32_t z, const float* psi) {
    if (flags & y) { slot[0][row][lane] = psi[0]; slot[5][row][lane] = psi[5]; }
    if (flags & z) { slot[1][row][lane] = psi[1]; slot[3][row][lane] = psi[3]; }
    if (flags & kLayerX) { slot[2][row][lane] = psi[2]; slot[4][row][lane] = psi[4]; }
  };
  auto kept_psi = [&](const float (*slot)[kMarchRows][kMarchCols], uint32_t y, uint32_t z, float* psi) {
    if (flags & y) { psi[0] = slot[0][row][lane]; psi[5] = slot[5][row][lane]; }
    if (flags & z) { psi[1] = slot[1][row][lane]; psi[3] = slot[3][row][lane]; }
    if (flags & kLayerX) { psi[2] = slot[2][row][lane]; psi[4] = slot[4][row][lane]; }
  };
  // running DFT of E over plane i: the steps n (`e1`) and, at T = 2, n + 1 (`e2`)
  auto full_dft = [&](int i, const V3& e1, const V3& e2) {
    if (!jn_ok) return;  // another tile's row; lanes of other tiles read (clamped) and do not write
    const MarchPtr f = fresh(a);
    const int nf = f->nf_dft;
    const uint64_t nxs = (uint64_t)snn * (nx - 1), nys = (uint64_t)smn * nx, nzs = (uint64_t)snm * nx;
    const float* w0c = f->dft_cos + (int64_t)n * nf;
    const float* w0s = f->dft_sin + (int64_t)n * nf;
    const bool dx = jn_ok && kn_ok && i < nx - 1, dy = jm_ok && kn_ok, dz = jn_ok && km_ok;
    auto add = [&](float s, float v1, float v2, float w1, float w2) {
      s = __builtin_fmaf(v1, w1, s);
      return T == 2 ? __builtin_fmaf(v2, w2, s) : s;
    };
    uint64_t ox = pm(i) * snn + rnn, oy = pn(i) * smn + rmn, oz = pn(i) * snm + rnm;
    // the sums of a few frequencies are read together before any of them is written:
    // one wait for memory per group, not per frequency (85^3, three frequencies, 100
    // steps: 4065 -> 3756 us; groups of four spill registers)
    for (int q0 = 0; q0 < nf; q0 += kMarchDft) {
      float r[kMarchDft][3], m[kMarchDft][3];
#pragma unroll
      for (int b = 0; b < kMarchDft; ++b) {
        if (q0 + b >= nf) continue;
        r[b][0] = row_load(f->dft_re[0] + (ox + b * nxs), kn4); m[b][0] = row_load(f->dft_im[0] + (ox + b * nxs), kn4);
        r[b][1] = row_load(f->dft_re[1] + (oy + b * nys), kn4); m[b][1] = row_load(f->dft_im[1] + (oy + b * nys), kn4);
        r[b][2] = row_load(f->dft_re[2] + (oz + b * nzs), km4); m[b][2] = row_load(f->dft_im[2] + (oz + b * nzs), km4);
      }
#pragma unroll
      for (int b = 0; b < kMarchDft; ++b) {
        const int q = q0 + b;
        if (q >= nf) continue;
        const float c1 = C(w0c)[q], s1 = C(w0s)[q];
        const float c2 = T == 2 ? C(w0c)[nf + q] : 0.0f, s2 = T == 2 ? C(w0s)[nf + q] : 0.0f;
        if (dx) {
          row_store(f->dft_re[0] + (ox + b * nxs), kn4, add(r[b][0], e1.x, e2.x, c1, c2));
          row_store(f->dft_im[0] + (ox + b * nxs), kn4, add(m[b][0], e1.x, e2.x, s1, s2));
        }
        if (dy) {
          row_store(f->dft_re[1] + (oy + b * nys), kn4, add(r[b][1], e1.y, e2.y, c1, c2));
          row_store(f->dft_im[1] + (oy + b * nys), kn4, add(m[b][1], e1.y, e2.y, s1, s2));
        }
        if (dz) {
          row_store(f->dft_re[2] + (oz + b * nzs), km4, add(r[b][2], e1.z, e2.z, c1, c2));
          row_store(f->dft_im[2] + (oz + b * nzs), km4, add(m[b][2], e1.z, e2.z, s1, s2));
        }
      }
      ox += kMarchDft * nxs;
      oy += kMarchDft * nys;
      oz += kMarchDft * nzs;
    }
  };

  // spacings and x planes that the march meets
  if (const int q = lane + kMarchCols * row; q < p1 + 2 - p0) {
    sh.ihx[q] = C(a->g.inv_h[0])[pm(p0 + q)];
    sh.iex[q] = C(a->g.inv_e[0])[pn(p0 + q)];
    uint32_t m = 0u;
    for (int o = 0; o < a->n_planes; ++o)
      if (a->planes[o].axis == 0 && a->planes[o].index == p0 + q) m |= 1u << o;
    sh.planes_x[q] = m;
  }
  lds_barrier();

  const V3 zero{0.0f, 0.0f, 0.0f};
  // E, H and curl coefficients of plane i, planes beyond the grid clamped
  auto load_e = [&](int i) {
    const MarchPtr f = fresh(a);
    return V3{row_load(f->in.e[0] + (pm(i) * snn + rnn), kn4), row_load(f->in.e[1] + (pn(i) * smn + rmn), kn4),
              row_load(f->in.e[2] + (pn(i) * snm + rnm), km4)};
  };
  auto load_h = [&](int i) {
    const MarchPtr f = fresh(a);
    return V3{row_load(f->in.h[0] + (pn(i) * smm + rmm), km4), row_load(f->in.h[1] + (pm(i) * snm + rnm), km4),
              row_load(f->in.h[2] + (pm(i) * smn + rmn), kn4)};
  };
  // the samples' byte offsets in plane p, by (rows, columns); the plane loop adds a
  // plane's size to each, and the arguments' moved buffers do the rest
  uint32_t onn = 4u * ((uint32_t)p0 * snn + rnn) + kn4, omn = 4u * ((uint32_t)p0 * smn + rmn) + kn4,
           onm = 4u * ((uint32_t)p0 * snm + rnm) + km4, omm = 4u * ((uint32_t)p0 * smm + rmm) + km4;
  V3 e = load_e(p0), en = load_e(p0 + 1), h = load_h(p0);
  V3 kc = COEF == 2 ? curl_value : load_curl(p0), kd = zero, kc1 = kc, kc2 = kc, kd2 = zero;  // planes p, p-1, p-2
  if (COEF == 0) kd = load_decay(p0);
  auto store_h = [&](bool im, const V3& v) {
    const MarchPtr f = fresh(a);
    if (km_ok) {
      if (jm_ok) row_store(f->behind_h[0], omm, v.x);
      if (jn_ok && im) row_store(f->behind_h[1], onm, v.y);
    }
    if (jm_ok && im && kn_ok) row_store(f->behind_h[2], omn, v.z);
  };
  auto store_e = [&](bool im, const V3& v) {
    const MarchPtr f = fresh(a);
    if (kn_ok) {
      if (jn_ok && im) row_store(f->behind_e[0], onn, v.x);
      if (jm_ok) row_store(f->behind_e[1], omn, v.y);
    }
    if (jn_ok && km_ok) row_store(f->behind_e[2], onm, v.z);
  };
  float ph[6] = {0, 0, 0, 0, 0, 0}, pe[6] = {0, 0, 0, 0, 0, 0};
  if (met & kLayers) load_psi(p0, ph, pe);
  // term samples of the planes that iteration p updates
  auto next_terms = [&](int p) {
#pragma unroll
    for (int q = 0; q < 2; ++q) tv_l[q][0] = tv_l[q][1] = 0.0f;
    if (ht.count == 1) sheet(0, p, p - 1, tv_l[0]);
    if (et.count == 1) sheet(1, p, p - 2, tv_l[1]);
  };
  next_terms(p0);
  auto take_terms = [&]() {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int t = 0; t < T; ++t) tv[q][t] = tv_l[q][t];
  };
  memory_settled();
  take_terms();
  V3 h1p = zero;              // H^{n+1/2} of plane p-1
  V3 a1 = zero, a2 = zero;    // E^{n+1} of planes p-1, p-2
  V3 b2 = zero, b3 = zero;    // H^{n+3/2} of planes p-2, p-3
  for (int p = p0; p <= p1; ++p) {
    flags = (uint32_t)held((int)met);
    const bool s1 = p <= first_last;
    // next plane's loads
    V3 e_l = zero, h_l = zero, kc_l = COEF == 2 ? curl_value : zero, kd_l = zero, kc2_l = zero, kd2_l = zero;
    if (p < first_last) {
      if (p <= steady) {
        const MarchPtr f = fresh(a);
        e_l = V3{row_load(f->ahead[0], onn), row_load(f->ahead[1], omn), row_load(f->ahead[2], onm)};
        h_l = V3{row_load(f->ahead[3], omm), row_load(f->ahead[4], onm), row_load(f->ahead[5], omn)};
        if (COEF == 1) kc_l = V3{row_load(f->ahead[6], onn), row_load(f->ahead[7], omn), row_load(f->ahead[8], onm)};
      } else {
        e_l = load_e(p + 2);
        h_l = load_h(p + 1);
        if (COEF == 1) kc_l = load_curl(p + 1);
      }
      if (COEF == 0) {
        kc_l = load_curl(p + 1);
        kd_l = load_decay(p + 1);
      }
    }
    float ph_l[6] = {0, 0, 0, 0, 0, 0}, pe_l[6] = {0, 0, 0, 0, 0, 0};
    if ((flags & kLayers) && p < first_last) load_psi(p + 1, ph_l, pe_l);
    next_terms(p + 1);
    if (T == 2 && COEF == 0 && p - 1 >= i0) {
      kc2_l = load_curl(p - 1);
      kd2_l = load_decay(p - 1);
    }
    sh.e1x[row][lane] = e.x;
    sh.e1z[row][lane] = e.z;
    if (T == 2) {
      sh.e2x[row][lane] = a1.x;
      sh.e2z[row][lane] = a1.z;
      sh.h2x[row][lane] = b2.x;
      sh.h2z[row][lane] = b2.z;
    }
    lds_barrier();
    if (p > p0 && slots > 0) store_z(p - 1);
    const float ex_j = sh.e1x[up][lane], ez_j = sh.e1z[up][lane];
    float ax_j = 0.0f, az_j = 0.0f;
    V3 h1 = zero, e1 = zero, h2 = zero, e2 = zero;
    if (s1) {
      h1 = update_h(p, 0, sh.ihx[p - p0], e, ex_j, ez_j, en, h, ph);
      if (T == 2 && (flags & kLayers)) keep_psi(sh.qh + 6 * (p & 1), kLayerHy, kLayerHz, ph);
    }
    sh.h1x[row][lane] = h1.x;
    sh.h1z[row][lane] = h1.z;
    const bool out_e = T == 2 ? p - 2 >= i0 : p >= i0;  // plane p-2 / p of E is this block's
    float q2e[6] = {0, 0, 0, 0, 0, 0}, q2h[6] = {0, 0, 0, 0, 0, 0};  // psi of the second step, E of p - 2 and H of p - 1
    if (T == 2) {
      ax_j = sh.e2x[up][lane];
      az_j = sh.e2z[up][lane];
      if (out_e) {
        if (flags & kLayers) kept_psi(sh.qe + 6 * (p & 1), kLayerEy, kLayerEz, q2e);
        e2 = update_e(p - 2, 1, sh.iex[p - 2 - p0], b2, sh.h2x[down][lane], sh.h2z[down][lane], b3.y, b3.z, a2, kc2,
                      kd2, q2e);
      }
    }
    lds_barrier();
    if (s1) {
      e1 = update_e(p, 0, sh.iex[p - p0], h1, sh.h1x[down][lane], sh.h1z[down][lane], h1p.y, h1p.z, e, kc, kd, pe);
      if (T == 2 && (flags & kLayers)) keep_psi(sh.qe + 6 * (p & 1), kLayerEy, kLayerEz, pe);
    }
    const bool out_h = T == 2 && p - 1 >= i0 && p - 1 < i1;
    if (T == 2 && p > p0 && p - 1 < i1) {
      if (flags & kLayers) kept_psi(sh.qh + 6 * ((p - 1) & 1), kLayerHy, kLayerHz, q2h);
      h2 = update_h(p - 1, 1, sh.ihx[p - 1 - p0], a1, ax_j, az_j, e1, h1p, q2h);
    }
    // the loads have had the whole plane to arrive; the plane's stores follow
    memory_settled();
    // the running sums are read ahead of the plane's stores, which retire in order
    if (DFT && out_e) full_dft(T == 2 ? p - 2 : p, T == 2 ? a2 : e1, T == 2 ? e2 : e1);
    if (T == 1 && out_e) {
      store_h(p < nx1, h1);
      store_e(p < nx1, e1);
      if (flags & (kLayerHy | kLayerHz | kLayerX)) store_psi_h(p, ph);
      if (flags & (kLayerEy | kLayerEz | kLayerX)) store_psi_e(p, pe);
    }
    if (T == 2 && out_e) {
      store_e(p - 2 < nx1, e2);
      if (flags & (kLayerEy | kLayerEz | kLayerX)) store_psi_e(p - 2, q2e);
    }
    if (out_h) {
      store_h(p - 1 < nx1, h2);
      if (flags & (kLayerHy | kLayerHz | kLayerX)) store_psi_h(p - 1, q2h);
    }
    if (T == 2 && out_e && (flags & kWatch)) observe(1, p - 2, e2, b2);
    if ((flags & kWatch) && s1 && p >= i0 && p < i1) observe(0, p, e1, h1);
    if (T == 2) {
      b3 = b2;
      b2 = h2;
      a2 = a1;
      a1 = e1;
      if (COEF == 1) {
        kc2 = kc1;
        kc1 = kc;
      }
      if (COEF == 0) {
        kc2 = kc2_l;
        kd2 = kd2_l;
      }
    }
    h1p = h1;
    e = en;
    en = e_l;
    h = h_l;
    kc = kc_l;
    kd = kd_l;
    onn += 4u * snn;
    omn += 4u * smn;
    onm += 4u * snm;
    omm += 4u * smm;
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      ph[q] = ph_l[q];
      pe[q] = pe_l[q];
    }
    take_terms();
  }
  if (slots > 0) {
    lds_barrier();
    store_z(p1);
  }
}

// Tile order: the hardware hands block w to XCD w % 8; each XCD gets a contiguous
// run of tiles (z fastest, then y), so tiles that share halo rows share an L2.
__device__ __forceinline__ int march_logical(int w, int blocks) { return (w % 8) * (blocks / 8) + w / 8; }

template <int T, int COEF, bool DFT>
__global__ __launch_bounds__(kMarchCols* kMarchRows) void march_kernel(MarchArgs args, int n) {
  __shared__ MarchShared<T> sh;
#ifdef MW_EMULATED_BLOCKS
  const MarchPtr a = &args;
#else
  const MarchPtr a = (MarchPtr)__builtin_amdgcn_kernarg_segment_ptr();  // `args` in place
#endif
  const int logical = march_logical((int)blockIdx.x, (int)gridDim.x);
  if (logical >= a->blocks) return;
  march_block<T, COEF, DFT>(a, n, logical, sh);
}

// One thread's share of a step of the TFSF line, H then (after a barrier) E; its
// states before each half step go to `he` / `hh` for the terms that sample them.
__device__ __forceinline__ void march_line_h(const mw_aux_line& line, float* he, float* hh, int m) {
#pragma clang fp contract(off)
  he[m] = line.e[m];
  if (m >= line.n_e - 1) return;
  const float de = line.e[m + 1] - line.e[m];
  const float v = __builtin_fmaf(-line.curl_h[m], de, line.decay_h[m] * line.h[m]);
  line.h[m] = v;
  hh[m] = v;
}
__device__ __forceinline__ void march_line_e(const mw_aux_line& line, int step, int m) {
#pragma clang fp contract(off)
  if (m == line.n_e - 1) line.e[m] = 0.0f;
  else if (m == 0) line.e[0] = line.source[step];
  else line.e[m] = __builtin_fmaf(-line.curl_e[m], line.h[m] - line.h[m - 1], line.decay_e[m] * line.e[m]);
}

// What a march of `steps` steps from step n needs beforehand, in one launch: block
// row y < set.count fills term y's time-shifted values of each of the steps; row
// set.count (one block) takes the TFSF line through them, leaving its states in
// `history` (E^n, H^{n+1/2}, E^{n+1}, H^{n+3/2}) for the terms that sample it.
__global__ __launch_bounds__(256) void march_prepare_kernel(TermSet set, mw_aux_line line, float* history, int n,
                                                            int steps, double dt) {
  const int q = blockIdx.y;
  if (q < set.count) {
    const mw_term& t = set.t[q];
    const int64_t cells = (int64_t)t.shape[0] * t.shape[1] * t.shape[2];
    const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= cells * steps) return;
    const int s = (int)(l / cells);
    const int64_t p = l - s * cells;
    const double time = (double)(n + s) * dt + t.t_offset - t.delay[p];
    t.values[l] = (float)(waveform(t.wave_kind, time, t.frequency, t.fwidth, t.amplitude, t.phase, t.delay0) *
                          (double)t.patch[p]);
    return;
  }
  if (blockIdx.x != 0 || line.n_e <= 0) return;
  for (int s = 0; s < steps; ++s) {
    float* he = history + (int64_t)(2 * s) * line.n_e;
    for (int m = threadIdx.x; m < line.n_e; m += blockDim.x) march_line_h(line, he, he + line.n_e, m);
    __syncthreads();
    for (int m = threadIdx.x; m < line.n_e; m += blockDim.x) march_line_e(line, n + s, m);
    __syncthreads();
  }
}

// Folds `rows` staged steps of the point observers into their sums, one thread per
// (frequency, point), in step order: the same bits wherever a run is split.
__global__ void march_points_kernel(const float* stage, int64_t row_floats, int rows, int n_points, int nf,
                                    const int32_t* component, const float* e_cos, const float* e_sin,
                                    const float* h_cos, const float* h_sin, float* re, float* im) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= n_points * nf) return;
  const int q = l % n_points, f = l / n_points;
  const float* wc = component[q] < 3 ? e_cos : h_cos;
  const float* ws = component[q] < 3 ? e_sin : h_sin;
  float c = re[l], s = im[l];
  for (int t = 0; t < rows; ++t) {
    const float v = stage[t * row_floats + q];
    c = __builtin_fmaf(v, wc[t * nf + f], c);
    s = __builtin_fmaf(v, ws[t * nf + f], s);
  }
  re[l] = c;
  im[l] = s;
}

}  // namespace mw
