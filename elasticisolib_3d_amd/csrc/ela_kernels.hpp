// Device kernels of the elastic isotropic 3-D propagator for gfx950.
//
// Scheme (reference: elastic_iso_float/src/kernelsElaGpu_3D.cu):
//   3-level leapfrog on 9 fields (vx vy vz sxx syy szz sxz sxy syz), 8th-order
//   staggered derivatives, cosine sponge. The reference runs, per fine step,
//   one stepper launch (kernelsElaGpu_3D.cu:110-460), 7 injection launches, a
//   damping launch over both time levels (:1182-1226) and 7 recording launches.
//   Here one fine step is one launch (velocity and stress blocks, which read
//   only level n and so are independent, and blocks that record level n; short
//   lists of sources are injected by the stencil's blocks, longer ones by a
//   launch behind it), with the sponge folded into the stencil:
//       n = w * (w * o + M D(c) [+ secondary source])
//   where every stored level has been damped exactly once. This equals the
//   reference's "step, inject, damp p0 and p1, swap" sequence, whose p0 after
//   the swap is the previous level damped a second time.
//
// Mapping to the CDNA4 execution model:
//   - a block owns a tile of 64 (z, one wave, coalesced) x 4, 8 or 16 (x)
//     cells, or of 32 x 8, which it marches along y over a chunk of planes;
//   - fields needing x or z derivatives are staged per plane in LDS with a
//     4-cell halo; y derivatives come from an 8-deep register queue per
//     thread, so each plane of each field is read from HBM once per tile;
//   - blocks are dealt round-robin to the 8 XCDs by the hardware, which sweeps
//     the grid; the default order hands out groups of whole z columns that way,
//     so that z and x neighbours share an L2 (orders: tile_coord).
// No MFMA: the stencil is not a dense contraction; the kernels are HBM-bound.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ela {

constexpr int FAT = 4;
constexpr int WAVE = 64;
constexpr int TZ = 64;       // z extent of the wide tiles = one wavefront

// Tile shapes S: 4, 8 and 16 are wide tiles of 64 (z) x S (x) cells, a wave
// covering one x row; TILE_NARROW is 32 x 8 cells, a wave covering two x rows
// of 32 (one 128-byte FP32 line each). Which grids
// take them, and what it measured, stands at narrow_tiles.
constexpr int TILE_NARROW = 32 + 8;
constexpr int tile_z(int S) { return S == TILE_NARROW ? 32 : TZ; }
constexpr int tile_x(int S) { return S == TILE_NARROW ? 8 : S; }
constexpr int tile_threads(int S) { return tile_z(S) * tile_x(S); }
constexpr int wave_rows(int S) { return WAVE / tile_z(S); }   // x rows per wave
constexpr int NXCD = 8;      // MI355X: 8 XCDs, blocks dealt round-robin

enum { VX = 0, VY, VZ, SXX, SYY, SZZ, SXZ, SXY, SYZ };
enum { BX_ = 0, BY_, BZ_, L2M, LAM, MXZ, MXY, MYZ };

// Stepper modes. The transposed steps (stepAdjGpuBorn_3D, n = w(w o - D (M c)),
// which multiplies by the medium at every loaded position,
// kernelsElaGpu_3D.cu:864-1040) read M c as the step before wrote it, one array
// per field as in the forward step.
enum { MODE_FWD = 0,       // n = w(w o + M D c)        stepFwdGpu_3D
       MODE_ADJ = 1,       // n = w(w o - M D c)        stepAdjGpu_3D
       MODE_BORN_ADJ_PM = 3, // n = w(w o - D q) with q = M c read and M n written (qn) beside n
       MODE_BORN_ADJ_Q = 4,  // the same on q = M n alone but for the normal stresses: q' = w(w q - M D c) (adj_wave)
       MODE_BORN_ADJ_MIXED = 5 // a stack of windows: _Q in the solid ones, _PM in the others (k_step)
};
constexpr bool premultiplied(int mode) { return mode >= MODE_BORN_ADJ_PM; }   // injections go into M n too

// Optional work fused into a stepper launch (bit flags).
//
// F_ACC and F_GRAD read and rewrite up to 18 and 8 arrays for values the step
// has in registers anyway: the new level n+1 and, in o, the level n-1 it
// replaces. So they run in every other step only and take both levels (pair;
// the schedule is pair_role), which halves that traffic:
//   Born transposed step: 75 -> 57 arrays a step on average (Born adjoint of
//   232x328x324, 40 steps: 105 -> 80 ms, the clearing of the targets gone too),
//   gradient transposed step: 64 -> 56 arrays (gradient of 232x328x324, 40
//   steps: 110 -> 108 ms).
enum { F_SS = 1,     // add the secondary sources ssl/ssr (Born forward)
       F_ACC = 2,    // accumulate the new level into accl/accr (coarse-time interpolation)
       F_STORE = 4,  // write the step's derivative combinations to dst (gradient recomputation)
       F_GRAD = 8,   // gradient imaging: grad[m] += new level x stored derivatives drv
       F_MED3 = 16,  // MODE_FWD / MODE_ADJ: form the 8 staggered, scaled medium values from (rho, lambda, mu)
       F_Q16 = 32    // FP32 with F_STORE / F_GRAD: the derivative combinations as block-scaled int16 (dq16, dqs)
};

// Derivative combinations stored as int16 (F_Q16): one scale per block of
// DQ_BLOCK values, the block being one 128-byte FP32 line of a z row, i.e.
// one half of a tile row's wave (rows and tiles start on a line), so that
// the scale of element i is dqs[i / DQ_BLOCK] for the steppers and the point
// kernels alike. q = rint(x / s), s = max |x| / 32767 over the block; the
// value restored is q s, within s / 2 (2^-16 of the block's largest value).
constexpr int DQ_BLOCK = 32;

// Every family of arrays is one buffer with the handle's array stride np, so
// an argument is its first array; array k of a family is fam(base, k, np).
// Inside the march np comes from an asm the compiler cannot see through: it
// forms each address where it is used (two scalar instructions) instead of
// keeping up to 60 pointers in scalar registers, whose spills took vector
// registers and, read back every plane, vector instructions.
template <typename T>
struct StepArgs {
  T* o;                 // level n-1 in, level n+1 out (in place)
  const T* c;           // level n
  const T* m;           // scaled medium
  const T* ssl;         // secondary sources (left / right coarse slices)
  const T* ssr;
  T* accl;              // coarse-time accumulation targets
  T* accr;
  T* dst;               // F_STORE: sx sy sz exx eyy ezz gxz gxy gyz of this step
  const T* drv;         // F_GRAD: the same combinations stored by the matching forward step
  T* grad;              // F_GRAD: gradient accumulators, one per medium array
  const T* q;           // MODE_BORN_ADJ_PM: M c of the current level
  T* qn;                // MODE_BORN_ADJ_PM: M n of the new level (written); MODE_BORN_ADJ_Q: n of the 3 normal stresses
  const T* ep;          // F_MED3: rho, lambda, mu
  int16_t* dq16;        // F_Q16: int16 derivative combinations (written by F_STORE, read by F_GRAD)
  float* dqs;           // F_Q16: their scales, one per DQ_BLOCK elements
  int64_t np;           // elements between the arrays of a family
  T tdt;                // F_MED3: 2 dtw
  double tdt64;         // F_MED3: 2 dtw in FP64 (FP32 steppers form buoyancies and normal moduli in FP64)
  T ssfl, ssfr;         // filter weights for the secondary source
  T accfl, accfr;       // filter weights for the accumulation
  T acc2l, acc2r;       // F_ACC with pair: those of the level in o
  const T* drv2;        // F_GRAD with pair: the derivative combinations of the level in o
  const int16_t* dq16b; // F_GRAD | F_Q16 with pair: the same as int16
  const float* dqsb;
  int pair;             // accumulate / image the level in o (n-1, complete) as well as the new one
  int accfirst;         // F_ACC: the left (1) or right (2) target holds nothing yet: written, not read
  T cx[4], cy[4], cz[4];
  const T* taper;       // [min_pad]
  int min_pad;
  int nz, nx, ny;       // grid sizes (reference layout)
  int nzi, zoff;        // internal row pitch and z origin (line-aligned interior)
  int64_t ys;           // nx * nzi
  int ychunk;
  int nbz, nbx, nby;    // tile counts along z, x, y-chunks
  int first;            // first tile of the launch: 0, or the tile count (stress blocks alone)
  int remap;            // tile order (see tile_coord)
  int rev;              // velocity blocks run backwards through the tiles (see k_step)
  int xgroup;           // x columns per group of the y-major order
  const int* chunks;    // stacked windows: per y chunk {y0, y1, window y0, window ny, window nx, window}, or null
  const int* fluid;     // MODE_BORN_ADJ_MIXED: per window, 1 general (_PM) or 0 solid (_Q)
};

template <typename P>
__device__ __forceinline__ P* fam(P* base, int k, int64_t np) { return base + k * np; }

__device__ __forceinline__ int64_t opaque(int64_t v) {
  asm volatile("" : "+s"(v));
  return v;
}

__device__ __forceinline__ int xcd_remap(int bid, int nb) {
  const int per = nb / NXCD, rem = nb % NXCD;
  const int xcd = bid % NXCD, k = bid / NXCD;
  return xcd < rem ? xcd * (per + 1) + k : rem * (per + 1) + (xcd - rem) * per + k;
}

// Groups of `gs` consecutive tiles dealt whole to one XCD: the k-th block that
// XCD x receives runs tile ((k / gs) * NXCD + x) * gs + k % gs, so the tiles
// running at one time still form one contiguous range of the enumeration (as
// in the hardware order) but each group's halo lines meet in one L2. Blocks
// past the last full round of NXCD groups keep the identity mapping.
__device__ __forceinline__ int xcd_group(int bid, int nb, int gs) {
  const int full = nb / (NXCD * gs) * (NXCD * gs);
  if (bid >= full) return bid;
  const int x = bid % NXCD, k = bid / NXCD;
  return ((k / gs) * NXCD + x) * gs + k % gs;
}

// Sponge factor from the distance to the nearest face of the cell's grid (or
// of its window when several windows are stacked along y).
template <typename T>
__device__ __forceinline__ T damp_w(const StepArgs<T>& a, int iz, int ix, int iy, int wy0, int wny, int wnx) {
  int d = min(min(iz - FAT, ix - FAT), min(a.nz - iz - 1 - FAT, wnx - ix - 1 - FAT));
  d = min(d, min(iy - wy0 - FAT, wy0 + wny - iy - 1 - FAT));
  return d < a.min_pad ? a.taper[d] : T(1);
}

// y-derivative from an 8-deep queue q[j] = f[iy - s + j], s = 3 for D+ and 4
// for D-: both reduce to sum_k c_k (q[4+k] - q[3-k]).
template <typename T>
__device__ __forceinline__ T dq(const T* q, const T* c) {
  return c[0] * (q[4] - q[3]) + c[1] * (q[5] - q[2]) + c[2] * (q[6] - q[1]) + c[3] * (q[7] - q[0]);
}

// LDS plane with a 4-cell halo on both sides in x (rows) and z (columns).
template <typename T, int S>
using Plane = T[tile_x(S) + 2 * FAT][tile_z(S) + 2 * FAT];

// D+ / D- along z (columns) and x (rows) of an LDS plane, at (r, col) = (ty+4, tz+4).
template <typename T, int S>
__device__ __forceinline__ T dpz(const Plane<T, S>& p, int r, int q, const T* c) {
  return c[0] * (p[r][q + 1] - p[r][q]) + c[1] * (p[r][q + 2] - p[r][q - 1]) +
         c[2] * (p[r][q + 3] - p[r][q - 2]) + c[3] * (p[r][q + 4] - p[r][q - 3]);
}
template <typename T, int S>
__device__ __forceinline__ T dmz(const Plane<T, S>& p, int r, int q, const T* c) {
  return c[0] * (p[r][q] - p[r][q - 1]) + c[1] * (p[r][q + 1] - p[r][q - 2]) +
         c[2] * (p[r][q + 2] - p[r][q - 3]) + c[3] * (p[r][q + 3] - p[r][q - 4]);
}
template <typename T, int S>
__device__ __forceinline__ T dpx(const Plane<T, S>& p, int r, int q, const T* c) {
  return c[0] * (p[r + 1][q] - p[r][q]) + c[1] * (p[r + 2][q] - p[r - 1][q]) +
         c[2] * (p[r + 3][q] - p[r - 2][q]) + c[3] * (p[r + 4][q] - p[r - 3][q]);
}
template <typename T, int S>
__device__ __forceinline__ T dmx(const Plane<T, S>& p, int r, int q, const T* c) {
  return c[0] * (p[r][q] - p[r - 1][q]) + c[1] * (p[r + 1][q] - p[r - 2][q]) +
         c[2] * (p[r + 2][q] - p[r - 3][q]) + c[3] * (p[r + 3][q] - p[r - 4][q]);
}

// Guard past the end of every library array (unpredicated stencil loads).
constexpr int GUARD_ROWS = 16;      // >= the largest tile_x
constexpr int GUARD_EXTRA = 2 * TZ;  // >= one tile height plus its z halo

// 32-bit element offsets from a uniform base pointer: the compiler can use
// the scalar-base + 32-bit vector-offset addressing mode, which saves the
// 64-bit per-lane address arithmetic. The host guarantees that every array
// is smaller than 4 GiB (ela_create checks n * sizeof(T) < 2^32).
template <typename T>
__device__ __forceinline__ const T* at(const T* base, uint32_t i) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + (uint64_t)(i * (uint32_t)sizeof(T)));
}
template <typename T>
__device__ __forceinline__ T* at(T* base, uint32_t i) {
  return reinterpret_cast<T*>(reinterpret_cast<char*>(base) + (uint64_t)(i * (uint32_t)sizeof(T)));
}
// Streaming accesses (read once / written once per step). The non-temporal
// cache policy is selectable at build time; measured on MI355X it slows the
// stencil down when applied to the loads, so loads default to the normal
// policy.
#ifndef ELA_NT_LOADS
#define ELA_NT_LOADS 0
#endif
#ifndef ELA_NT_STORES
#define ELA_NT_STORES 1
#endif
template <typename T>
__device__ __forceinline__ T ld_nt(const T* base, uint32_t i) {
#if ELA_NT_LOADS
  return __builtin_nontemporal_load(at(base, i));
#else
  return *at(base, i);
#endif
}
template <typename T>
__device__ __forceinline__ void st_nt(T* base, uint32_t i, T v) {
#if ELA_NT_STORES
  __builtin_nontemporal_store(v, at(base, i));
#else
  *at(base, i) = v;
#endif
}

// FP32 LDS rows loaded straight from HBM (1) or staged through registers (0).
#ifndef ELA_LDS_DMA
#define ELA_LDS_DMA 1
#endif

// Direct global -> LDS load of one row of a tile (FP32): lane l of the wave
// writes row[l], so a 64-lane wave fills TZ consecutive LDS values without
// passing them through registers. Completion is covered by the wait that
// precedes the block's next barrier.
__device__ __forceinline__ void row_to_lds(const float* base, uint32_t i, float* row) {
  __builtin_amdgcn_global_load_lds(at(base, i), (__attribute__((address_space(3))) void*)row, 4, 0, 0);
}

// The rows of a tile plane that a wave loads: plane[row][col ...] and, of a
// narrow tile, plane[row + 1][col ...] by the upper half of the lanes (lane l
// writes 4 l bytes past the row given, hence the shift by half a wave). The
// two comments in the assembly keep the compiler from merging the branches
// into one load whose LDS row, a wave-uniform operand, would be the lower
// half's for every lane.
template <int S, typename P>
__device__ __forceinline__ void rows_to_lds(const float* base, uint32_t i, P& plane, int row, int col) {
  if constexpr (wave_rows(S) == 1) {
    row_to_lds(base, i, &plane[row][col]);
  } else {
    if (threadIdx.x < WAVE / 2) {
      row_to_lds(base, i, &plane[row][col]);
      asm volatile("; lower lanes");
    } else {
      row_to_lds(base, i, &plane[row + 1][col] - WAVE / 2);
      asm volatile("; upper lanes");
    }
  }
}

// Largest magnitude over each 32-lane half of the wave (one DQ_BLOCK), in
// every lane: DPP lane moves inside each 16-lane row (swap neighbours, swap
// pairs, mirror within 8, mirror within 16) and one swizzle that exchanges
// the two rows of a half (lane ^ 16). Each half must be active or inactive as a
// whole (a narrow tile's second x row may lie past the interior) and no move may
// cross the halves. The magnitudes are compared as unsigned integers (the bit patterns of
// non-negative floats order as their values), which needs no NaN quieting.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_umax(uint32_t u) {
  return max(u, (uint32_t)__builtin_amdgcn_mov_dpp((int)u, CTRL, 0xF, 0xF, true));
}

__device__ __forceinline__ float half_wave_absmax(float x) {
  uint32_t u = __float_as_uint(fabsf(x));
  u = dpp_umax<0xB1>(u);   // quad_perm [1, 0, 3, 2]
  u = dpp_umax<0x4E>(u);   // quad_perm [2, 3, 0, 1]
  u = dpp_umax<0x141>(u);  // row_half_mirror
  u = dpp_umax<0x140>(u);  // row_mirror
  u = max(u, (uint32_t)__builtin_amdgcn_ds_swizzle((int)u, 0x401F));  // lane ^ 16
  return __uint_as_float(u);
}

// F_Q16 store of one derivative combination at element i: every lane of an
// interior x row (half a wave of a narrow tile) calls it; lanes past the row's
// interior cells pass x = 0. The last z tile of a
// row may reach past the row into the next row's leading non-interior line
// ([0, zoff + FAT) = [0, 32)), which no stepper reads and no other tile
// writes. The hardware reciprocal (1 ulp) serves for 1 / m: |x| 32767 rcp(m)
// stays below 32767.5, so q fits int16, and the stored scale is what the
// reader multiplies by, so the error stays within s / 2 plus a few FP32 ulps.
__device__ __forceinline__ void store_dq16(int16_t* q, float* sc, uint32_t i, float x) {
  const float m = half_wave_absmax(x);
  const float inv = m > 0.f ? 32767.f * __builtin_amdgcn_rcpf(m) : 0.f;
  st_nt(q, i, (int16_t)__float2int_rn(x * inv));
  if ((threadIdx.x & (DQ_BLOCK - 1)) == 0) *at(sc, i / DQ_BLOCK) = m * (1.f / 32767.f);
}

__device__ __forceinline__ float load_dq16(const int16_t* q, const float* sc, uint32_t i) {
  return (float)*at(q, i) * *at(sc, i / DQ_BLOCK);
}

// The stencil's loads are not predicated: a tile's columns, halo rows and halo
// column past the grid are clamped to its last row and column (tile_coord),
// where no interior cell's stencil reads them. That keeps them inside the
// arrays and makes idle lanes read lines their neighbours read anyway
// (unclamped, behind every array's guard of GUARD_ROWS rows plus GUARD_EXTRA
// elements, forward 152x152x148 took 5 % longer).

// Per-thread tile geometry, halo roles and 32-bit column offsets.
//
// Internal layout: rows of nzi elements (a multiple of one 128-byte cache
// line) with the reference's z = 0 stored at zoff, chosen so that the first
// interior cell (z = FAT) starts a cache line; a 64-wide tile then covers
// exactly two (FP32) lines and its z halos are the adjacent lines.
struct TileCoord {
  int tz, ty, iz, izo, ix, y0, y1, z0, x0;   // iz internal, izo reference z
  int wy0, wny, wnx;       // the tile's window: first plane, planes, x extent (whole grid without windows)
  int win;                 // its number
  bool empty;              // no interior cell in the tile (its window is narrower than the tile's x)
  bool active;             // own column inside the interior
  bool xin;                // the tile row (a wave, half a wave of a narrow tile) is an interior x row
  bool xh, zh;             // x-halo loader (ty < 4), z-halo loader (tz < 8)
  int colh;                // LDS column of the z-halo value
  uint32_t col, cxl, cxh, czh;  // own column, x-halo rows, z-halo column, each clamped to the grid (window)
  uint32_t colu;                // own column, not clamped (F_Q16 stores of whole lines)
};

// Block -> tile. order 0: the hardware's dealing (block b runs on XCD b % 8)
// over tiles enumerated z fastest, then x, then y. order 1: each XCD gets a
// contiguous range of that enumeration. order 2: contiguous ranges of a
// y-major enumeration (per z tile, groups of `xgroup` x columns, y chunks
// within a group, columns fastest), so that the blocks an XCD runs at the
// same time are y- and x-neighbours whose halo planes meet in its L2.
// order 3: the z-fastest enumeration dealt to the XCDs in groups of whole z
// columns (`xgroup` adjacent columns of nbz tiles), so that z (and, with
// xgroup > 1, x) neighbours share an L2 while the grid is swept in the
// hardware order.
template <int S>
__device__ __forceinline__ TileCoord tile_coord(int bid, int nbz, int nbx, int nby, int ychunk, int nz, int nzi,
                                                int zoff, int nx, int ny, int order, int xgroup, const int* chunks) {
  constexpr int BX = tile_x(S), BZ = tile_z(S);
  const int nb = nbz * nbx * nby;
  const int lb = order == 3 ? xcd_group(bid, nb, nbz * xgroup) : order ? xcd_remap(bid, nb) : bid;
  int bz, bx, by;
  if (order == 2) {
    const int per_z = nbx * nby;
    bz = lb / per_z;
    const int p = lb - bz * per_z;
    const int grp = p / (xgroup * nby);
    const int r = p - grp * xgroup * nby;
    const int width = min(xgroup, nbx - grp * xgroup);
    by = r / width;
    bx = grp * xgroup + (r - by * width);
  } else {
    bz = lb % nbz;
    bx = (lb / nbz) % nbx;
    by = lb / (nbz * nbx);
  }
  TileCoord t;
  t.tz = wave_rows(S) == 1 ? threadIdx.x : threadIdx.x % BZ;
  t.ty = wave_rows(S) == 1 ? threadIdx.y : threadIdx.y * wave_rows(S) + threadIdx.x / BZ;
  t.z0 = zoff + FAT + bz * BZ;
  t.x0 = FAT + bx * BX;
  t.iz = t.z0 + t.tz;
  t.izo = t.iz - zoff;
  t.ix = t.x0 + t.ty;
  if (chunks) {
    const int* c = chunks + 8 * by;
    t.y0 = c[0]; t.y1 = c[1]; t.wy0 = c[2]; t.wny = c[3]; t.wnx = c[4]; t.win = c[5];
  } else {
    t.y0 = FAT + by * ychunk;
    t.y1 = min(t.y0 + ychunk, ny - FAT);
    t.wy0 = 0; t.wny = ny; t.wnx = nx; t.win = 0;
  }
  nx = t.wnx;
  t.empty = t.x0 >= nx - FAT;
  t.xin = t.ix < nx - FAT;
  t.active = (t.izo < nz - FAT) && t.xin;
  t.xh = t.ty < FAT;
  const int ixlo = t.x0 - FAT + t.ty, ixhi = t.x0 + BX + t.ty;
  t.zh = t.tz < 2 * FAT;
  const int izh = t.tz < FAT ? t.z0 - FAT + t.tz : t.z0 + BZ + (t.tz - FAT);
  t.colh = t.tz < FAT ? t.tz : BZ + t.tz;
  // Lanes past the last z cell and rows past the last x row read the last
  // one: no interior stencil uses their values, and without the clamp they
  // fetched lines nobody needs (a 144-cell z interior is 2.25 tiles: 200
  // steps on the 152 x 152 x 148 grid 23.3 -> 22.2 ms, 201 x 187 x 143 22.0
  // -> 21.4 ms; no change where the interior fills its tiles).
  const int izc = min(t.iz, zoff + nz - 1), ixc = min(t.ix, nx - 1);
  t.col = (uint32_t)(ixc * nzi + izc);
  t.cxl = (uint32_t)(min(ixlo, nx - 1) * nzi + izc);
  t.cxh = (uint32_t)(min(ixhi, nx - 1) * nzi + izc);
  t.czh = (uint32_t)(ixc * nzi + min(izh, zoff + nz - 1));
  t.colu = (uint32_t)(t.ix * nzi + t.iz);
  return t;
}

// ---------------------------------------------------------------------------
// Sparse points: injection and recording of all 9 components.
// ---------------------------------------------------------------------------
template <typename T>
struct PointArgs {
  const int32_t* pos[9];   // internal-layout positions of the component's grid (-1: skip)
  int64_t n[9];
  int64_t off[10];         // prefix offsets over components
  T* field[9];             // wavefield component arrays
  T* tr[9];                // traces
  int64_t tr_stride_pt;    // element stride between points in tr (nts for [n][nts], 1 for [nts][n])
  int64_t tr_stride_t;     // element stride between time samples (1 for [n][nts], n for [nts][n])
  int its;
  T fa, fb;                // filter weights for its and its+1
  // optional coarse accumulation of the injected value (Born passes)
  T* accl[9];
  T* accr[9];
  T accfl, accfr;
  // optional gradient imaging of the injected value (adjoint-state gradient);
  // with dq16 set the derivative combinations are the F_Q16 int16 arrays
  const T* drv[9];
  const int16_t* dq16[9];
  const float* dqs[9];
  T* grad[8];
  // optional premultiplied level to keep consistent (MODE_BORN_ADJ_PM)
  T* q[9];
  const T* m[8];
  // damping (injection only)
  const T* taper;
  int min_pad, nz, nx, ny, nzi, zoff;
  const int* ytab;         // stacked windows: per plane {window y0, window ny, window nx, window}, or null
  const int* fluid;        // per window: general steps (1) or MODE_BORN_ADJ_Q (0), or null: field says it
  const int* its_dev;      // coarse sample index read from device memory (graph replays), or null
  int its_off;             // added to the index read from its_dev
  // fine step k = *step_dev + step_off read from device memory (graph replays
  // of gradient steps), or null: the coarse sample is k / sub and the weights
  // are filt[i + fo] and filt[sub + 1 + i + fo] with i = k % sub (the host's
  // fa / fb of that step)
  const int* step_dev;
  const T* filt;
  int sub, fo, step_off;
  int nmax;                // > 0: a launch whose coarse sample (its_dev) or fine step (step_dev) is outside
                           // [0, nmax) does nothing (the recording of a level before the first or after the last)
  const int* box;          // box of the points (see inject_tile), for an injection fused into a step
};

// Coarse sample and time-filter weights of a point launch; false: outside the record.
// (PA: PointArgs<T>, or the same in the kernel argument segment, see inject_tile.)
template <typename T, typename PA>
__device__ __forceinline__ bool point_time(const PA& a, int& its, T& fa, T& fb) {
  if (a.step_dev) {
    const int k = *a.step_dev + a.step_off;
    if (a.nmax && (k < 0 || k >= a.nmax)) return false;
    its = k / a.sub;
    const int i = k - its * a.sub + a.fo;
    fa = a.filt[i];
    fb = a.filt[a.sub + 1 + i];
  } else {
    its = a.its_dev ? *a.its_dev + a.its_off : a.its;
    if (a.its_dev && a.nmax && (its < 0 || its >= a.nmax)) return false;
    fa = a.fa;
    fb = a.fb;
  }
  return true;
}

template <typename T>
__device__ __forceinline__ int comp_of(const PointArgs<T>& a, int64_t g) {
  int c = 0;
#pragma unroll
  for (int k = 1; k < 9; ++k) c += (g >= a.off[k]) ? 1 : 0;
  return c;
}

template <typename T, typename PA>
__device__ __forceinline__ T point_taper(const PA& a, int32_t p) {
  const int ys = a.nzi * a.nx;
  const int iy = p / ys;
  const int rem = p - iy * ys;
  const int ix = rem / a.nzi;
  const int iz = rem - ix * a.nzi - a.zoff;
  int wy0 = 0, wny = a.ny, wnx = a.nx;
  if (a.ytab) { wy0 = a.ytab[4 * iy]; wny = a.ytab[4 * iy + 1]; wnx = a.ytab[4 * iy + 2]; }
  int d = min(min(iz - FAT, ix - FAT), min(a.nz - iz - 1 - FAT, wnx - ix - 1 - FAT));
  d = min(d, min(iy - wy0 - FAT, wy0 + wny - iy - 1 - FAT));
  return d < a.min_pad ? a.taper[d] : T(1);
}

// field[pos] += w(pos) * (tr[its] fa + tr[its+1] fb)
// (ker_inject_source_* / ker_inject_data_*, kernelsElaGpu_3D.cu:11-52, with the
// sponge factor that the reference applies right after injection).
// Roundings are fixed (no contraction but the written fma), so that the
// fused and the separate injection give the same bits.
template <typename T, bool ACC, bool GRAD, bool PM, typename PA>
__device__ __forceinline__ void inject_point(const PA& a, int c, int64_t k) {
#pragma clang fp contract(off)
  const int32_t p = a.pos[c][k];
  int its;
  T fa, fb;
  (void)point_time<T>(a, its, fa, fb);
  const T taper = point_taper<T>(a, p);
  // the injected value of component cc at this point (the three normal
  // stresses share their point list, so index k is the same point for them)
  auto injected = [&](int cc) {
    const T* tr = a.tr[cc] + k * a.tr_stride_pt;
    return taper * fma(tr[(int64_t)its * a.tr_stride_t], fa, tr[(int64_t)(its + 1) * a.tr_stride_t] * fb);
  };
  const T v = injected(c);
  if (!PM || a.field[c]) a.field[c][p] += v;  // MODE_BORN_ADJ_Q: the normal stresses alone hold n
  if (ACC && a.accl[c]) {
    a.accl[c][p] += v * a.accfl;
    a.accr[c][p] += v * a.accfr;
  }
  // Points are unique within a component's list, so every update below has
  // one writer; the normal stresses, coupled through lamb2MuDtw / lambDtw,
  // are updated together by the sxx thread, with the stepper's formulas.
  T vn[3] = {T(0), T(0), T(0)};
  if ((PM || GRAD) && c == SXX) { vn[0] = v; vn[1] = injected(SYY); vn[2] = injected(SZZ); }
  if (PM) {
    // keep q = M n
    if (c < 3) {
      a.q[c][p] += v * a.m[c][p];
    } else if (c == SXX) {
      const T l2 = a.m[L2M][p], la = a.m[LAM][p];
      a.q[SXX][p] += vn[0] * l2 + (vn[1] + vn[2]) * la;
      a.q[SYY][p] += vn[1] * l2 + (vn[0] + vn[2]) * la;
      a.q[SZZ][p] += vn[2] * l2 + (vn[0] + vn[1]) * la;
    } else if (c >= SXZ) {
      a.q[c][p] += v * a.m[MXZ + (c - SXZ)][p];
    }
  }
  if (GRAD) {
    // the stepper imaged the level before this injection; add the injected part
    auto drv = [&](int cc) -> T {
      return a.dq16[cc] ? T(load_dq16(a.dq16[cc], a.dqs[cc], (uint32_t)p)) : a.drv[cc][p];
    };
    if (c < 3) {
      a.grad[c][p] += v * drv(c);
    } else if (c == SXX) {
      const T dxx = drv(SXX), dyy = drv(SYY), dzz = drv(SZZ);
      const T l2 = vn[0] * dxx + vn[1] * dyy + vn[2] * dzz;
      a.grad[L2M][p] += l2;
      a.grad[LAM][p] += (vn[0] + vn[1] + vn[2]) * (dxx + dyy + dzz) - l2;
    } else if (c >= SXZ) {
      a.grad[MXZ + (c - SXZ)][p] += v * drv(c);
    }
  }
}

// n = M^-1 q of a velocity or shear component of MODE_BORN_ADJ_Q. Not
// contracted with what forms m, so that a loaded medium and one formed in the
// step give the same bits.
template <typename T>
__device__ __forceinline__ T level_of(T q, T m) {
#pragma clang fp contract(off)
  return q * (T(1) / m);
}

// tr[its] += field[pos] fa ; tr[its+1] += field[pos] fb
// (ker_record_interp_data_* / ker_record_source_*, kernelsElaGpu_3D.cu:61-104).
template <typename T>
__device__ __forceinline__ void record_point(const PointArgs<T>& a, int64_t g) {
  if (g >= a.off[9]) return;
  const int c = comp_of(a, g);
  const int64_t k = g - a.off[c];
  const int32_t p = a.pos[c][k];
  if (p < 0) return;
  int its;
  T fa, fb;
  if (!point_time<T>(a, its, fa, fb)) return;
  // MODE_BORN_ADJ_Q holds no n of the velocities and shear stresses
  bool held = a.field[c] != nullptr;
  if (a.fluid && (c < SXX || c > SZZ)) held = a.fluid[a.ytab[4 * (p / (a.nzi * a.nx)) + 3]];
  const T v = held ? a.field[c][p] : level_of(a.q[c][p], a.m[c < 3 ? c : MXZ + (c - SXZ)][p]);
  T* tr = a.tr[c] + k * a.tr_stride_pt;
  T& t0 = tr[(int64_t)its * a.tr_stride_t];
  T& t1 = tr[(int64_t)(its + 1) * a.tr_stride_t];
  t0 = fma(v, fa, t0);
  t1 = fma(v, fb, t1);
}

// Injection by a step's own blocks: after its march a block whose tile meets
// the points' box adds the listed points inside its tile (components c0 ..
// c1 - 1, those the block has written) with inject_point, so that a step with
// few sources is one launch. The barrier orders the block's stores of the new
// level before the read-modify-writes; no other block touches these cells.
// With the recording moved into the step after (step_with_points) that took
// 40x36x44, 100 steps through host arrays, from 1.68 to 1.17 ms, 152x152x148
// (200 steps) from 20.1 to 18.6 ms and 328x472x468 with 2.9 M recorded points
// (80 steps) from 143.0 to 138.9 ms.
//
// box: the largest of (POS_TOP - z, z, POS_TOP - x, x, POS_TOP - y, y) over
// the points, in internal z, so that a zeroed box holds nothing. It is tested
// during the prologue, where its load hides behind the stencil's (40x36x44: 8.16 -> 7.97 us a step).
constexpr int POS_TOP = 1 << 30;

template <typename T, int S>
__device__ __forceinline__ bool box_hit(const PointArgs<T>& a, const TileCoord& t) {
  if (a.off[9] == 0) return false;
  const int* b = a.box;
  return POS_TOP - b[0] < t.z0 + tile_z(S) && b[1] >= t.z0 && POS_TOP - b[2] < t.x0 + tile_x(S) && b[3] >= t.x0 &&
         POS_TOP - b[4] < t.y1 && b[5] >= t.y0;
}

// Everything is read again from the kernel's argument segment (k_step's
// second argument is the injection) through an address the compiler cannot
// trace back, and the tile worked out again from the block index: kept live
// across the march they cost scalar registers, whose spills take vector
// registers (130 instead of 128, i.e. 3 waves per SIMD, in some steps).
template <typename T, int S, bool ACC, bool GRAD, bool PM>
__device__ __forceinline__ void inject_tile(int half, int c0, int c1) {
#define ELA_KERNARG __attribute__((address_space(4)))
  uint64_t seg = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(seg));
  const auto& s = *(const ELA_KERNARG StepArgs<T>*)seg;
  const auto& a = *(const ELA_KERNARG PointArgs<T>*)(seg + sizeof(StepArgs<T>));
#undef ELA_KERNARG
  const int nb = s.nbz * s.nbx * s.nby, b0 = (int)blockIdx.x + s.first, bid = half ? b0 - nb : s.rev ? nb - 1 - b0 : b0;
  const TileCoord t = tile_coord<S>(bid, s.nbz, s.nbx, s.nby, s.ychunk, s.nz, s.nzi, s.zoff, s.nx, s.ny, s.remap, s.xgroup, s.chunks);
  constexpr int BX = tile_x(S), BZ = tile_z(S);
  __syncthreads();
  for (int g = (int)a.off[c0] + t.ty * BZ + t.tz; g < (int)a.off[c1]; g += BZ * BX) {
    int c = c0;
#pragma nounroll   // one offset at a time in a scalar register
    for (int k = c0 + 1; k < c1; ++k) c += g >= (int)a.off[k] ? 1 : 0;
    const int64_t k = g - a.off[c];
    const int32_t p = a.pos[c][k];
    if (p < 0) continue;
    const int row = p / a.nzi, z = p - row * a.nzi, y = row / a.nx, x = row - y * a.nx;
    if (z >= t.z0 && z < t.z0 + BZ && x >= t.x0 && x < t.x0 + BX && y >= t.y0 && y < t.y1)
      inject_point<T, ACC, GRAD, PM>(a, c, k);
  }
}

// ---------------------------------------------------------------------------
// Velocity update: vx, vy, vz from the six stresses.
//
// Software pipeline per y plane: the global loads of plane iy+1 (new queue
// values, LDS centres and halos) are issued before plane iy is computed and
// land in the second LDS buffer, so one barrier per plane suffices and the
// HBM latency overlaps the stencil arithmetic.
// ---------------------------------------------------------------------------
// The velocity stepper's LDS: double-buffered planes of sxx, szz, sxy, sxz,
// syz and (F_MED3) density planes with the low x row and low z column.
template <typename T, int S, bool MED3>
struct VelLds {
  Plane<T, S> xx[2], zz[2], xy[2], xz[2], yz[2];
  T rho[2][MED3 ? tile_x(S) + 1 : 1][MED3 ? tile_z(S) + 1 : 1];
};

template <typename T>
struct VelStage {
  T xx, zz, xz;                 // LDS centres of the non-queue fields
  T hxx0, hxx1, hxy0, hxy1, hxz0, hxz1;  // x-halo rows (low / high)
  T hzz, hxz, hyz;              // z-halo column
  T nxy, nyy, nyz;              // new queue values (plane + 4, + 3, + 4)
  T rho, rho_hx, rho_hz;        // F_MED3: density of the column, of row x0 - 1 and of z0 - 1
};

// F_MED3: the staggered, scaled medium formed in the stepper from (rho,
// lambda, mu) with the interior rule of the host scaling (a cell's staggered
// value averages it with its lower neighbour along the axis; the FD interior
// never meets the edge rules): rhox = (rho + rho[x-1]) / 2, rhoxDtw = 2 dtw /
// rhox (likewise y, z); lamb2MuDtw = 2 dtw (lambda + 2 mu), lambDtw = 2 dtw
// lambda; muxzDtw = 2 dtw * Sz(Sx(mu)) with S the same half-cell average, muxy
// = Sy(Sx(mu)), muyz = Sz(Sy(mu)) -- the operations of ela_scale_medium in the
// same order, so an FP64 stepper reproduces the 8-array stepper exactly.
//
// Buoyancy 2 dtw / rho_h of a staggered density rho_h. FP64: the host
// scaling's division. FP32: the same correctly rounded FP64 division of the
// FP64 half-cell sum of the FP32 densities, rounded once to FP32 -- the host's
// FP64 scaling of the same densities rounded to FP32, bit for bit. Formed in
// FP32 arithmetic, the buoyancies and moduli carried one or two extra
// roundings whose bias more than doubled the FP32 data's distance from FP64
// over a 5000-step run. k_scale_medium uses the same functions, so every mode
// of one handle sees the same medium.
template <typename T>
__device__ __forceinline__ T buoy_h(T tdt, double tdt64, double rho_h) {
  if constexpr (sizeof(T) == 4) {
    return T(tdt64 / rho_h);
  } else {
    return tdt / T(rho_h);
  }
}

template <typename T>
__device__ __forceinline__ T stag_buoy(const StepArgs<T>& a, T c, T m) {
  if constexpr (sizeof(T) == 4) return buoy_h<T>(a.tdt, a.tdt64, 0.5 * (double(c) + double(m)));
  else return a.tdt / (T(0.5) * (c + m));
}

// lamb2MuDtw and lambDtw of a cell (FP32: formed in FP64, rounded once).
template <typename T>
__device__ __forceinline__ void normal_moduli(T tdt, double tdt64, T lam, T mu, T& l2m, T& la) {
  if constexpr (sizeof(T) == 4) {
    l2m = T(tdt64 * (double(lam) + 2.0 * double(mu)));
    la = T(tdt64 * double(lam));
  } else {
    l2m = tdt * (lam + T(2) * mu);
    la = tdt * lam;
  }
}

template <typename T, int S, int MODE, int F>
__device__ __forceinline__ void velocity_block(const StepArgs<T>& a, const PointArgs<T>& inj, int bid,
                                               VelLds<T, S, (F & F_MED3) != 0>& L) {
  constexpr int BX = tile_x(S);
  constexpr bool SS = (F & F_SS) != 0, ACC = (F & F_ACC) != 0, MED3 = (F & F_MED3) != 0;
  constexpr bool Q16 = (F & F_Q16) != 0, QS = Q16 && (F & F_STORE) != 0;
  static_assert(!Q16 || sizeof(T) == 4, "F_Q16 is an FP32 format");
  static_assert(!QS || (!SS && !ACC && (F & F_GRAD) == 0 && MODE == MODE_FWD), "F_Q16 stores: MODE_FWD recomputation");
  constexpr bool HOIST = sizeof(T) == 4;  // per-cell operands loaded ahead of the stores
  auto& l_xx = L.xx; auto& l_zz = L.zz; auto& l_xy = L.xy; auto& l_xz = L.xz; auto& l_yz = L.yz;
  auto& l_rho = L.rho;
  const TileCoord t = tile_coord<S>(bid, a.nbz, a.nbx, a.nby, a.ychunk, a.nz, a.nzi, a.zoff, a.nx, a.ny, a.remap, a.xgroup, a.chunks);
  if (t.empty) return;  // block-uniform, before any barrier
  const uint32_t ys = (uint32_t)a.ys;
  int64_t np = a.np;
  // FP32 rows go straight from HBM to LDS, FP64 rows through registers
  constexpr bool DMA = ELA_LDS_DMA && sizeof(T) == 4;
  auto src = [&](int f) -> const T* { return fam(MODE == MODE_BORN_ADJ_PM ? a.q : a.c, f, np); };
  auto val = [&](int f, uint32_t i) { return *at(src(f), i); };
  const int r = t.ty + FAT, q = t.tz + FAT;
  // first x row of the wave (a wide tile's wave is one row), wave-uniform
  const int wy = __builtin_amdgcn_readfirstlane(t.ty), wr = wy + FAT;

  // plane p's values: LDS rows of buffer nb directly (DMA), the rest into v
  auto fetch = [&](VelStage<T>& v, int p, int nb) {
    const uint32_t pl = (uint32_t)p * ys;
    if constexpr (DMA) {
      rows_to_lds<S>(src(SXX), pl + t.col, l_xx[nb], wr, FAT);
      rows_to_lds<S>(src(SZZ), pl + t.col, l_zz[nb], wr, FAT);
      rows_to_lds<S>(src(SXZ), pl + t.col, l_xz[nb], wr, FAT);
    } else {
      v.xx = val(SXX, pl + t.col);
      v.zz = val(SZZ, pl + t.col);
      v.xz = val(SXZ, pl + t.col);
    }
    v.nxy = val(SXY, pl + 4 * ys + t.col);
    v.nyy = val(SYY, pl + 3 * ys + t.col);
    v.nyz = val(SYZ, pl + 4 * ys + t.col);
    if (wy < FAT) {  // the x-halo loaders (t.xh) are whole waves
      if constexpr (DMA) {
        rows_to_lds<S>(src(SXX), pl + t.cxl, l_xx[nb], wy, FAT); rows_to_lds<S>(src(SXX), pl + t.cxh, l_xx[nb], wr + BX, FAT);
        rows_to_lds<S>(src(SXY), pl + t.cxl, l_xy[nb], wy, FAT); rows_to_lds<S>(src(SXY), pl + t.cxh, l_xy[nb], wr + BX, FAT);
        rows_to_lds<S>(src(SXZ), pl + t.cxl, l_xz[nb], wy, FAT); rows_to_lds<S>(src(SXZ), pl + t.cxh, l_xz[nb], wr + BX, FAT);
      } else {
        v.hxx0 = val(SXX, pl + t.cxl); v.hxx1 = val(SXX, pl + t.cxh);
        v.hxy0 = val(SXY, pl + t.cxl); v.hxy1 = val(SXY, pl + t.cxh);
        v.hxz0 = val(SXZ, pl + t.cxl); v.hxz1 = val(SXZ, pl + t.cxh);
      }
    }
    if (t.zh) {
      v.hzz = val(SZZ, pl + t.czh); v.hxz = val(SXZ, pl + t.czh); v.hyz = val(SYZ, pl + t.czh);
    }
    if (MED3) {
      // the column's own cell and its x - 1 / z - 1 neighbours
      if constexpr (DMA) {
        rows_to_lds<S>(fam(a.ep, 0, np), pl + t.col, l_rho[nb], wy + 1, 1);
        if (t.ty == 0) row_to_lds(fam(a.ep, 0, np), pl + t.col - (uint32_t)a.nzi, &l_rho[nb][0][1]);
      } else {
        v.rho = *at(fam(a.ep, 0, np), pl + t.col);
        if (t.ty == 0) v.rho_hx = *at(fam(a.ep, 0, np), pl + t.col - (uint32_t)a.nzi);
      }
      if (t.tz == 0) v.rho_hz = *at(fam(a.ep, 0, np), pl + t.col - 1u);
    }
  };
  // the values fetch kept in registers, and the queue centres
  auto stage = [&](int b, const VelStage<T>& v, T cxy, T cyz) {
    if constexpr (!DMA) { l_xx[b][r][q] = v.xx; l_zz[b][r][q] = v.zz; l_xz[b][r][q] = v.xz; }
    l_xy[b][r][q] = cxy; l_yz[b][r][q] = cyz;
    if (!DMA && t.xh) {
      l_xx[b][t.ty][q] = v.hxx0; l_xx[b][r + BX][q] = v.hxx1;
      l_xy[b][t.ty][q] = v.hxy0; l_xy[b][r + BX][q] = v.hxy1;
      l_xz[b][t.ty][q] = v.hxz0; l_xz[b][r + BX][q] = v.hxz1;
    }
    if (t.zh) { l_zz[b][r][t.colh] = v.hzz; l_xz[b][r][t.colh] = v.hxz; l_yz[b][r][t.colh] = v.hyz; }
    if (MED3) {
      if constexpr (!DMA) {
        l_rho[b][t.ty + 1][t.tz + 1] = v.rho;
        if (t.ty == 0) l_rho[b][0][t.tz + 1] = v.rho_hx;
      }
      if (t.tz == 0) l_rho[b][t.ty + 1][0] = v.rho_hz;
    }
  };
  // F_MED3: density of the column on the previous plane (y - 1)
  T rho_prev = MED3 ? *at(fam(a.ep, 0, np), (uint32_t)(t.y0 - 1) * ys + t.col) : T(0);

  // queues: sxy (D+y, q[j] = f[iy-3+j]), syy (D-y, f[iy-4+j]), syz (D+y)
  T qxy[8], qyy[8], qyz[8];
#pragma unroll
  for (int j = 0; j < 7; ++j) {
    qxy[j] = val(SXY, (uint32_t)(t.y0 - 3 + j) * ys + t.col);
    qyy[j] = val(SYY, (uint32_t)(t.y0 - 4 + j) * ys + t.col);
    qyz[j] = val(SYZ, (uint32_t)(t.y0 - 3 + j) * ys + t.col);
  }
  bool inj_hit;  // block-uniform
  {
    VelStage<T> v0;
    fetch(v0, t.y0, 0);
    qxy[7] = v0.nxy; qyy[7] = v0.nyy; qyz[7] = v0.nyz;
    inj_hit = box_hit<T, S>(inj, t);
    stage(0, v0, qxy[3], qyz[3]);
  }
  __syncthreads();
  int b = 0;
  for (int iy = t.y0; iy < t.y1; ++iy) {
    const bool more = iy + 1 < t.y1;
    np = opaque(a.np);
    VelStage<T> nx_;
    if (more) fetch(nx_, iy + 1, b ^ 1);  // buffer b ^ 1 is free: every wave passed the last barrier
    // F_STORE with F_Q16: all lanes of an interior row take the branch (the
    // block maxima are reductions over half waves) and the interior ones store
    if (QS ? t.xin : t.active) {
      const uint32_t i = (uint32_t)iy * ys + (QS ? t.colu : t.col);
      const T* cx = a.cx; const T* cy = a.cy; const T* cz = a.cz;
      // FP32: every per-cell operand is loaded before the first store (the
      // stores could alias them as far as the compiler knows, and a load
      // issued after a store waits for it); FP64 loads them where they are
      // used, which holds fewer registers (2 waves per SIMD)
      T o3[3], m3[3], ss3[3], al3[3], ar3[3], g3[3], d3[3], e3[3];
      auto load_ss = [&](int f) { return *at(fam(a.ssl, f, np), i) * a.ssfl + *at(fam(a.ssr, f, np), i) * a.ssfr; };
      auto load_acc = [&](int f) {
        al3[f] = a.accfirst == 1 ? T(0) : *at(fam(a.accl, f, np), i);
        ar3[f] = a.accfirst == 2 ? T(0) : *at(fam(a.accr, f, np), i);
      };
      auto load_grad = [&](int f) {  // BX_/BY_/BZ_ == VX/VY/VZ
        g3[f] = *at(fam(a.grad, f, np), i);
        if constexpr (Q16) d3[f] = load_dq16(fam(a.dq16, f, np), fam(a.dqs, f, np / DQ_BLOCK), i);
        else d3[f] = ld_nt(fam(a.drv, f, np), i);
        if (a.pair) {
          if constexpr (Q16) e3[f] = load_dq16(fam(a.dq16b, f, np), fam(a.dqsb, f, np / DQ_BLOCK), i);
          else e3[f] = ld_nt(fam(a.drv2, f, np), i);
        }
      };
      // the level n of a value of this step's arrays (MODE_BORN_ADJ_Q: they hold M n)
      auto level = [&](T v, int f) { return MODE == MODE_BORN_ADJ_Q ? level_of(v, m3[f]) : v; };
#pragma unroll
      for (int f = 0; f < 3; ++f) {
        o3[f] = ld_nt(fam(a.o, f, np), i);
        if (!MED3) m3[f] = ld_nt(fam(a.m, f, np), i);
        if constexpr (HOIST) {
          if (SS) ss3[f] = load_ss(f);
          if (ACC) load_acc(f);
          if (F & F_GRAD) load_grad(f);
        }
      }
      if (MED3) {
        const T rc = l_rho[b][t.ty + 1][t.tz + 1];
        m3[0] = stag_buoy(a, rc, l_rho[b][t.ty][t.tz + 1]);
        m3[1] = stag_buoy(a, rc, rho_prev);
        m3[2] = stag_buoy(a, rc, l_rho[b][t.ty + 1][t.tz]);
      }
      const T sx = dmx<T, S>(l_xx[b], r, q, cx) + dq(qxy, cy) + dpz<T, S>(l_xz[b], r, q, cz);
      const T sy = dpx<T, S>(l_xy[b], r, q, cx) + dq(qyy, cy) + dpz<T, S>(l_yz[b], r, q, cz);
      const T sz = dpx<T, S>(l_xz[b], r, q, cx) + dq(qyz, cy) + dmz<T, S>(l_zz[b], r, q, cz);
      T w = T(0);
      if (!QS || t.active) w = damp_w(a, t.izo, t.ix, iy, t.wy0, t.wny, t.wnx);
      const T s3[3] = {sx, sy, sz};
      if (F & F_STORE) {
#pragma unroll
        for (int f = 0; f < 3; ++f) {
          if constexpr (QS) store_dq16(fam(a.dq16, f, np), fam(a.dqs, f, np / DQ_BLOCK), i, t.active ? s3[f] : T(0));
          else st_nt(fam(a.dst, f, np), i, s3[f]);
        }
      }
#pragma unroll
      for (int f = 0; f < 3; ++f) {
        T u;
        if (MODE == MODE_FWD) u = w * o3[f] + m3[f] * s3[f];
        else if (MODE == MODE_ADJ || MODE == MODE_BORN_ADJ_Q) u = w * o3[f] - m3[f] * s3[f];
        else u = w * o3[f] - s3[f];
        if constexpr (!HOIST) {
          if (SS) ss3[f] = load_ss(f);
          if (ACC) load_acc(f);
          if (F & F_GRAD) load_grad(f);
        }
        if (SS) u += ss3[f];
        u *= w;
        if (QS && !t.active) continue;
        st_nt(fam(a.o, f, np), i, u);
        if (MODE == MODE_BORN_ADJ_PM) st_nt(fam(a.qn, f, np), i, u * m3[f]);
        if (ACC || (F & F_GRAD)) {
          const T n = level(u, f), n2 = a.pair ? level(o3[f], f) : T(0);
          if (ACC) {
            if (a.pair) { al3[f] += n2 * a.acc2l; ar3[f] += n2 * a.acc2r; }
            *at(fam(a.accl, f, np), i) = al3[f] + n * a.accfl;
            *at(fam(a.accr, f, np), i) = ar3[f] + n * a.accfr;
          }
          if (F & F_GRAD) {
            if (a.pair) g3[f] += n2 * e3[f];
            *at(fam(a.grad, f, np), i) = g3[f] + n * d3[f];
          }
        }
      }
    }
    if (MED3) rho_prev = l_rho[b][t.ty + 1][t.tz + 1];
#pragma unroll
    for (int j = 0; j < 7; ++j) { qxy[j] = qxy[j + 1]; qyy[j] = qyy[j + 1]; qyz[j] = qyz[j + 1]; }
    if (more) {
      qxy[7] = nx_.nxy; qyy[7] = nx_.nyy; qyz[7] = nx_.nyz;
      stage(b ^ 1, nx_, qxy[3], qyz[3]);
    }
    __syncthreads();
    b ^= 1;
  }
  if (inj_hit) inject_tile<T, S, ACC, (F & F_GRAD) != 0, premultiplied(MODE)>(0, VX, SXX);
}

// ---------------------------------------------------------------------------
// Stress update: six stresses from vx, vy, vz (same pipeline).
// ---------------------------------------------------------------------------
// The stress stepper's LDS: double-buffered planes of vx, vy, vz and (F_MED3)
// shear-modulus planes with the low x row and low z column.
template <typename T, int S, bool MED3>
struct StressLds {
  Plane<T, S> vx[2], vy[2], vz[2];
  T mu[2][MED3 ? tile_x(S) + 1 : 1][MED3 ? tile_z(S) + 1 : 1];
};

template <typename T>
struct StressStage {
  T hlo[3], hhi[3], hz[3];   // x-halo rows and z-halo column of vx, vy, vz
  T nx, ny, nz;              // new queue values (vx: plane+3, vy: +4, vz: +3)
  T mu, mu_hx, mu_hz, mu_hc; // F_MED3: shear modulus of the column, row x0 - 1, z0 - 1 and both
};

template <typename T, int S, int MODE, int F>
__device__ __forceinline__ void stress_block(const StepArgs<T>& a, const PointArgs<T>& inj, int bid,
                                             StressLds<T, S, (F & F_MED3) != 0>& L) {
  constexpr int BX = tile_x(S);
  constexpr bool SS = (F & F_SS) != 0, ACC = (F & F_ACC) != 0, MED3 = (F & F_MED3) != 0;
  constexpr bool Q16 = (F & F_Q16) != 0, QS = Q16 && (F & F_STORE) != 0;
  static_assert(!Q16 || sizeof(T) == 4, "F_Q16 is an FP32 format");
  static_assert(!QS || (!SS && !ACC && (F & F_GRAD) == 0 && MODE == MODE_FWD), "F_Q16 stores: MODE_FWD recomputation");
  constexpr bool HOIST = sizeof(T) == 4;  // per-cell operands loaded ahead of the stores
  auto& l_vx = L.vx; auto& l_vy = L.vy; auto& l_vz = L.vz; auto& l_mu = L.mu;
  const TileCoord t = tile_coord<S>(bid, a.nbz, a.nbx, a.nby, a.ychunk, a.nz, a.nzi, a.zoff, a.nx, a.ny, a.remap, a.xgroup, a.chunks);
  if (t.empty) return;  // block-uniform, before any barrier
  const uint32_t ys = (uint32_t)a.ys;
  int64_t np = a.np;
  constexpr bool DMA = ELA_LDS_DMA && sizeof(T) == 4;
  auto src = [&](int f) -> const T* { return fam(MODE == MODE_BORN_ADJ_PM ? a.q : a.c, f, np); };
  auto val = [&](int f, uint32_t i) { return *at(src(f), i); };
  const int r = t.ty + FAT, q = t.tz + FAT;
  const int wy = __builtin_amdgcn_readfirstlane(t.ty), wr = wy + FAT;  // wave-uniform row

  // plane p's values: LDS rows of buffer nb directly (DMA), the rest into v
  auto fetch = [&](StressStage<T>& v, int p, int nb) {
    const uint32_t pl = (uint32_t)p * ys;
    v.nx = val(VX, pl + 3 * ys + t.col);
    v.ny = val(VY, pl + 4 * ys + t.col);
    v.nz = val(VZ, pl + 3 * ys + t.col);
    if (wy < FAT) {  // the x-halo loaders (t.xh) are whole waves
      if constexpr (DMA) {
        rows_to_lds<S>(src(VX), pl + t.cxl, l_vx[nb], wy, FAT); rows_to_lds<S>(src(VX), pl + t.cxh, l_vx[nb], wr + BX, FAT);
        rows_to_lds<S>(src(VY), pl + t.cxl, l_vy[nb], wy, FAT); rows_to_lds<S>(src(VY), pl + t.cxh, l_vy[nb], wr + BX, FAT);
        rows_to_lds<S>(src(VZ), pl + t.cxl, l_vz[nb], wy, FAT); rows_to_lds<S>(src(VZ), pl + t.cxh, l_vz[nb], wr + BX, FAT);
      } else {
#pragma unroll
        for (int f = 0; f < 3; ++f) { v.hlo[f] = val(f, pl + t.cxl); v.hhi[f] = val(f, pl + t.cxh); }
      }
    }
    if (t.zh) {
#pragma unroll
      for (int f = 0; f < 3; ++f) v.hz[f] = val(f, pl + t.czh);
    }
  };
  // F_MED3: shear modulus of plane p around the column
  auto fetch_mu = [&](StressStage<T>& v, int p, int nb) {
    const uint32_t pl = (uint32_t)p * ys, nzi = (uint32_t)a.nzi;
    if constexpr (DMA) {
      rows_to_lds<S>(fam(a.ep, 2, np), pl + t.col, l_mu[nb], wy + 1, 1);
      if (t.ty == 0) row_to_lds(fam(a.ep, 2, np), pl + t.col - nzi, &l_mu[nb][0][1]);
    } else {
      v.mu = *at(fam(a.ep, 2, np), pl + t.col);
      if (t.ty == 0) v.mu_hx = *at(fam(a.ep, 2, np), pl + t.col - nzi);
    }
    if (t.tz == 0) v.mu_hz = *at(fam(a.ep, 2, np), pl + t.col - 1u);
    if (t.ty == 0 && t.tz == 0) v.mu_hc = *at(fam(a.ep, 2, np), pl + t.col - nzi - 1u);
  };
  auto stage_mu = [&](int m, const StressStage<T>& v) {
    if constexpr (!DMA) {
      l_mu[m][t.ty + 1][t.tz + 1] = v.mu;
      if (t.ty == 0) l_mu[m][0][t.tz + 1] = v.mu_hx;
    }
    if (t.tz == 0) l_mu[m][t.ty + 1][0] = v.mu_hz;
    if (t.ty == 0 && t.tz == 0) l_mu[m][0][0] = v.mu_hc;
  };
  // the values fetch kept in registers, and the queue centres
  auto stage = [&](int b, const StressStage<T>& v, T cvx, T cvy, T cvz) {
    l_vx[b][r][q] = cvx; l_vy[b][r][q] = cvy; l_vz[b][r][q] = cvz;
    if (!DMA && t.xh) {
      l_vx[b][t.ty][q] = v.hlo[0]; l_vx[b][r + BX][q] = v.hhi[0];
      l_vy[b][t.ty][q] = v.hlo[1]; l_vy[b][r + BX][q] = v.hhi[1];
      l_vz[b][t.ty][q] = v.hlo[2]; l_vz[b][r + BX][q] = v.hhi[2];
    }
    if (t.zh) { l_vx[b][r][t.colh] = v.hz[0]; l_vy[b][r][t.colh] = v.hz[1]; l_vz[b][r][t.colh] = v.hz[2]; }
  };

  // queues: vx (D-y, q[j] = f[iy-4+j]), vy (D+y, f[iy-3+j]), vz (D-y)
  T qx[8], qy[8], qz[8];
#pragma unroll
  for (int j = 0; j < 7; ++j) {
    qx[j] = val(VX, (uint32_t)(t.y0 - 4 + j) * ys + t.col);
    qy[j] = val(VY, (uint32_t)(t.y0 - 3 + j) * ys + t.col);
    qz[j] = val(VZ, (uint32_t)(t.y0 - 4 + j) * ys + t.col);
  }
  // F_MED3: the previous plane's terms carried in registers -- Sx(mu) of the
  // column, mu of the column and of its z - 1 neighbour -- which are the
  // current plane's values one iteration later (same operands, same order)
  T sx_prev = T(0), mu_prev = T(0), muz_prev = T(0);
  if (MED3) {
    const uint32_t pl = (uint32_t)(t.y0 - 1) * ys;
    mu_prev = *at(fam(a.ep, 2, np), pl + t.col);
    muz_prev = *at(fam(a.ep, 2, np), pl + t.col - 1u);
    sx_prev = T(0.5) * (mu_prev + *at(fam(a.ep, 2, np), pl + t.col - (uint32_t)a.nzi));
  }
  bool inj_hit;  // block-uniform
  {
    StressStage<T> v0;
    fetch(v0, t.y0, 0);
    qx[7] = v0.nx; qy[7] = v0.ny; qz[7] = v0.nz;
    inj_hit = box_hit<T, S>(inj, t);
    stage(0, v0, qx[4], qy[3], qz[4]);
    if (MED3) {
      fetch_mu(v0, t.y0, 0);
      stage_mu(0, v0);
    }
  }
  __syncthreads();
  int b = 0;
  for (int iy = t.y0; iy < t.y1; ++iy) {
    const bool more = iy + 1 < t.y1;
    np = opaque(a.np);
    StressStage<T> nx_;
    if (more) {  // buffer b ^ 1 is free: every wave passed the last barrier
      fetch(nx_, iy + 1, b ^ 1);
      if (MED3) fetch_mu(nx_, iy + 1, b ^ 1);
    }
    if (QS ? t.xin : t.active) {  // F_Q16 stores: see velocity_block
      const uint32_t i = (uint32_t)iy * ys + (QS ? t.colu : t.col);
      const T* cx = a.cx; const T* cy = a.cy; const T* cz = a.cz;
      // FP32: every per-cell operand is loaded before the first store (see velocity_block)
      T o6[6], ss6[6], al6[6], ar6[6], g5[5], d6[6], e6[6];
      auto load_ss = [&](int f) { return *at(fam(a.ssl, f, np), i) * a.ssfl + *at(fam(a.ssr, f, np), i) * a.ssfr; };
      T l2m = 0, lam = 0, mxz = 0, mxy = 0, myz = 0;
      auto load_acc = [&](int k) {
        const int f = SXX + k;
        al6[k] = a.accfirst == 1 ? T(0) : *at(fam(a.accl, f, np), i);
        ar6[k] = a.accfirst == 2 ? T(0) : *at(fam(a.accr, f, np), i);
      };
      // the level n of a value v of shear stress k (MODE_BORN_ADJ_Q holds M n)
      auto level = [&](T v, int k) {
        if constexpr (MODE == MODE_BORN_ADJ_Q) return level_of(v, k == 3 ? mxz : k == 4 ? mxy : myz);
        else return v;
      };
      // g5 += the image of level v with the derivative combinations d:
      // lamb2MuDtw multiplies exx, eyy, ezz in sxx, syy, szz; lambDtw the
      // other two normal strains; the shear moduli one shear strain each
      auto image_normal = [&](const T* v, const T* d) {
        const T l2 = v[0] * d[0] + v[1] * d[1] + v[2] * d[2];
        g5[0] += l2;
        g5[1] += (v[0] + v[1] + v[2]) * (d[0] + d[1] + d[2]) - l2;
      };
      auto image_shear = [&](const T* v, const T* d) {
#pragma unroll
        for (int k = 3; k < 6; ++k) g5[k - 1] += level(v[k], k) * d[k];
      };
      auto load_g = [&]() {
#pragma unroll
        for (int m = 0; m < 5; ++m) g5[m] = *at(fam(a.grad, L2M + m, np), i);
      };
      auto load_e = [&]() {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          if constexpr (Q16) e6[k] = load_dq16(fam(a.dq16b, SXX + k, np), fam(a.dqsb, SXX + k, np / DQ_BLOCK), i);
          else e6[k] = ld_nt(fam(a.drv2, SXX + k, np), i);
        }
      };
      auto load_d = [&]() {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          if constexpr (Q16) d6[k] = load_dq16(fam(a.dq16, SXX + k, np), fam(a.dqs, SXX + k, np / DQ_BLOCK), i);
          else d6[k] = ld_nt(fam(a.drv, SXX + k, np), i);
        }
      };
      // the arrays of the level that is replaced
      auto level_at = [&](int k) {
        return MODE == MODE_BORN_ADJ_Q && k < 3 ? fam(a.qn, k, np) : fam(a.o, SXX + k, np);
      };
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        o6[k] = ld_nt(level_at(k), i);
        if constexpr (HOIST) {
          if (SS) ss6[k] = load_ss(SXX + k);
          if (ACC) load_acc(k);
        }
      }
      if constexpr (HOIST && (F & F_GRAD) != 0) {
        load_g();
        if (a.pair) {
          load_e();
          image_normal(o6, e6);
          if constexpr (MODE != MODE_BORN_ADJ_Q) image_shear(o6, e6);  // else below, with the medium
        }
        load_d();
      }
      if (MED3) {
        const int rr = t.ty + 1, qq = t.tz + 1;
        const T mu_c = l_mu[b][rr][qq], mu_xm = l_mu[b][rr - 1][qq], mu_zm = l_mu[b][rr][qq - 1];
        const T mu_xzm = l_mu[b][rr - 1][qq - 1];
        const T lr = ld_nt(fam(a.ep, 1, np), i);
        normal_moduli(a.tdt, a.tdt64, lr, mu_c, l2m, lam);
        const T sx_c = T(0.5) * (mu_c + mu_xm), sx_zm = T(0.5) * (mu_zm + mu_xzm);
        const T sy_c = T(0.5) * (mu_c + mu_prev), sy_zm = T(0.5) * (mu_zm + muz_prev);
        mxz = (T(0.5) * (sx_c + sx_zm)) * a.tdt;
        mxy = (T(0.5) * (sx_c + sx_prev)) * a.tdt;
        myz = (T(0.5) * (sy_c + sy_zm)) * a.tdt;
      } else {
        l2m = ld_nt(fam(a.m, L2M, np), i); lam = ld_nt(fam(a.m, LAM, np), i);
        mxz = ld_nt(fam(a.m, MXZ, np), i); mxy = ld_nt(fam(a.m, MXY, np), i); myz = ld_nt(fam(a.m, MYZ, np), i);
      }
      const T exx = dpx<T, S>(l_vx[b], r, q, cx);
      const T eyy = dq(qy, cy);
      const T ezz = dpz<T, S>(l_vz[b], r, q, cz);
      const T gxy = dq(qx, cy) + dmx<T, S>(l_vy[b], r, q, cx);
      const T gxz = dmz<T, S>(l_vx[b], r, q, cz) + dmx<T, S>(l_vz[b], r, q, cx);
      const T gyz = dq(qz, cy) + dmz<T, S>(l_vy[b], r, q, cz);
      T w = T(0);
      if (!QS || t.active) w = damp_w(a, t.izo, t.ix, iy, t.wy0, t.wny, t.wnx);
      if (F & F_STORE) {
        if constexpr (QS) {
          const T e6[6] = {exx, eyy, ezz, gxz, gxy, gyz};
#pragma unroll
          for (int k = 0; k < 6; ++k) store_dq16(fam(a.dq16, SXX + k, np), fam(a.dqs, SXX + k, np / DQ_BLOCK), i, t.active ? e6[k] : T(0));
        } else {
          st_nt(fam(a.dst, SXX, np), i, exx); st_nt(fam(a.dst, SYY, np), i, eyy); st_nt(fam(a.dst, SZZ, np), i, ezz);
          st_nt(fam(a.dst, SXZ, np), i, gxz); st_nt(fam(a.dst, SXY, np), i, gxy); st_nt(fam(a.dst, SYZ, np), i, gyz);
        }
      }
      T u[6];
      if (MODE == MODE_BORN_ADJ_PM || MODE == MODE_BORN_ADJ_Q) {
        u[0] = w * o6[0] - exx;
        u[1] = w * o6[1] - eyy;
        u[2] = w * o6[2] - ezz;
      } else {
        const T sg = MODE == MODE_FWD ? T(1) : T(-1);
        u[0] = w * o6[0] + sg * (l2m * exx) + sg * (lam * (eyy + ezz));
        u[1] = w * o6[1] + sg * (l2m * eyy) + sg * (lam * (exx + ezz));
        u[2] = w * o6[2] + sg * (l2m * ezz) + sg * (lam * (exx + eyy));
      }
      if (MODE == MODE_BORN_ADJ_PM) {
        u[3] = w * o6[3] - gxz;
        u[4] = w * o6[4] - gxy;
        u[5] = w * o6[5] - gyz;
      } else {
        const T sg = MODE == MODE_FWD ? T(1) : T(-1);
        u[3] = w * o6[3] + sg * (mxz * gxz);
        u[4] = w * o6[4] + sg * (mxy * gxy);
        u[5] = w * o6[5] + sg * (myz * gyz);
      }
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const int f = SXX + k;
        if constexpr (!HOIST) {
          if (SS) ss6[k] = load_ss(f);
        }
        T v = u[k];
        if (SS) v += ss6[k];
        v *= w;
        u[k] = v;
        if (QS && !t.active) continue;
        st_nt(level_at(k), i, v);
      }
      if constexpr (ACC) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          const int f = SXX + k;
          const T n = k < 3 ? u[k] : level(u[k], k);
          if constexpr (!HOIST) load_acc(k);
          if (a.pair) {
            const T n2 = k < 3 ? o6[k] : level(o6[k], k);
            al6[k] += n2 * a.acc2l; ar6[k] += n2 * a.acc2r;
          }
          *at(fam(a.accl, f, np), i) = al6[k] + n * a.accfl;
          *at(fam(a.accr, f, np), i) = ar6[k] + n * a.accfr;
        }
      }
      if (MODE == MODE_BORN_ADJ_PM || MODE == MODE_BORN_ADJ_Q) {
        T* const qn = MODE == MODE_BORN_ADJ_Q ? a.o : a.qn;
        st_nt(fam(qn, SXX, np), i, u[0] * l2m + (u[1] + u[2]) * lam);
        st_nt(fam(qn, SYY, np), i, u[1] * l2m + (u[0] + u[2]) * lam);
        st_nt(fam(qn, SZZ, np), i, u[2] * l2m + (u[0] + u[1]) * lam);
      }
      if (MODE == MODE_BORN_ADJ_PM) {
        st_nt(fam(a.qn, SXZ, np), i, u[3] * mxz);
        st_nt(fam(a.qn, SXY, np), i, u[4] * mxy);
        st_nt(fam(a.qn, SYZ, np), i, u[5] * myz);
      }
      if (F & F_GRAD) {
        if constexpr (!HOIST) {
          load_g();
          if (a.pair) { load_e(); image_normal(o6, e6); }
        }
        if ((!HOIST || MODE == MODE_BORN_ADJ_Q) && a.pair) image_shear(o6, e6);
        if constexpr (!HOIST) load_d();
        image_normal(u, d6);
        image_shear(u, d6);
#pragma unroll
        for (int m = 0; m < 5; ++m) *at(fam(a.grad, L2M + m, np), i) = g5[m];
      }
    }
#pragma unroll
    for (int j = 0; j < 7; ++j) { qx[j] = qx[j + 1]; qy[j] = qy[j + 1]; qz[j] = qz[j + 1]; }
    if (MED3) {
      // this plane's terms become the previous plane's (every thread, active or not)
      const int rr = t.ty + 1, qq = t.tz + 1;
      mu_prev = l_mu[b][rr][qq];
      muz_prev = l_mu[b][rr][qq - 1];
      sx_prev = T(0.5) * (mu_prev + l_mu[b][rr - 1][qq]);
    }
    if (more) {
      qx[7] = nx_.nx; qy[7] = nx_.ny; qz[7] = nx_.nz;
      stage(b ^ 1, nx_, qx[4], qy[3], qz[4]);
      if (MED3) stage_mu(b ^ 1, nx_);
    }
    __syncthreads();
    b ^= 1;
  }
  if (inj_hit) inject_tile<T, S, ACC, (F & F_GRAD) != 0, premultiplied(MODE)>(1, SXX, SYZ + 1);
}

// ---------------------------------------------------------------------------
// One fine step: the velocity blocks, then the stress blocks, in one launch
// (both read level n only). Small grids are bound by the latency of a march
// (about 1.2 us a plane) and by the launch itself, which the two halves now
// share: 40x36x44 tile 8x4 20.5 -> 13.8 us a step with inject and record,
// 110x93x121 49.8 -> 43.4 us, 152x152x148 105.8 -> 96.9 us (FP32, tile 8x8,
// order 3/2). Large grids gain only the first half's tail (232x328x324 638.7
// -> 637.2 us, 328x472x468 1721.8 -> 1718.6 us): they are bound by HBM.
//
// With a.rev the velocity blocks run through the tiles backwards: the stress
// blocks of the launch before ended at the last tiles, and what they wrote and
// read there (sigma n, v n-1, 9 of the 13 arrays a velocity block touches) is
// still in the 256 MB Infinity Cache. Adjoint 232x328x324 64.9 -> 64.3 ms in one
// process and 64.7 -> 62.9 in another, Born adjoint 83.2 -> 78.1 ms; nothing at
// 152x152x148, which the cache does not limit. It costs the planes that a block
// shares with the y chunk after it, which then were read two layers of chunks
// ago instead of just now: launch_step_s reverses where four layers fit.
//
// MODE_BORN_ADJ_MIXED holds two forms of a block and takes that of the window
// its chunk belongs to (transposed steps of two windows 328x290x260, one with a
// fluid, half of them imaging: 1.76-1.79 ms a step against 1.84-1.88 in the
// general form alone; a launch for each form cost stacks of 60^3 windows 15 to
// 26 % of a backward pass).
// ---------------------------------------------------------------------------
// Waves per SIMD asked of the compiler: the FP32 steps without per-cell extra
// operands need 115-129 VGPRs and run at 4 (at most 128); the others hold more
// and take what they get (1: no request).
template <typename T, int FV, int FS>
constexpr int step_waves() {
  return sizeof(T) == 4 && ((FV | FS) & (F_SS | F_ACC | F_GRAD)) == 0 ? 4 : 1;
}

template <typename T, int S, int MODE, int FV, int FS>
__global__ void __launch_bounds__(tile_threads(S), (step_waves<T, FV, FS>())) k_step(StepArgs<T> a, PointArgs<T> inj, PointArgs<T> rec) {
  // one LDS object: the compiler's wait analysis then tells the rows the
  // direct loads fill (buffer b ^ 1) from the rows the stencil reads (buffer b)
  union Lds {
    VelLds<T, S, (FV & F_MED3) != 0> v;
    StressLds<T, S, (FS & F_MED3) != 0> s;
  };
  __shared__ Lds L;
  static_assert(sizeof(StepArgs<T>) % alignof(PointArgs<T>) == 0, "inject_tile finds inj behind a");
  const int nb = a.nbz * a.nbx * a.nby, bid = (int)blockIdx.x + a.first;  // block-uniform
  if (bid < 2 * nb) {
    const bool vel = bid < nb;
    const int tile = vel ? (a.rev ? nb - 1 - bid : bid) : bid - nb;
    if constexpr (MODE == MODE_BORN_ADJ_MIXED) {
      const int w = tile_coord<S>(tile, a.nbz, a.nbx, a.nby, a.ychunk, a.nz, a.nzi, a.zoff, a.nx, a.ny, a.remap,
                                  a.xgroup, a.chunks).win;
      if (a.fluid[w]) {
        if (vel) velocity_block<T, S, MODE_BORN_ADJ_PM, FV>(a, inj, tile, L.v);
        else stress_block<T, S, MODE_BORN_ADJ_PM, FS>(a, inj, tile, L.s);
      } else {
        StepArgs<T> s = a;   // q in the places of n, the normal stresses of n as adj_args hands them over
        s.o = a.qn;
        s.c = a.q;
        s.qn = fam(a.o, SXX, a.np);
        if (vel) velocity_block<T, S, MODE_BORN_ADJ_Q, FV>(s, inj, tile, L.v);
        else stress_block<T, S, MODE_BORN_ADJ_Q, FS>(s, inj, tile, L.s);
      }
    } else if (vel) {
      velocity_block<T, S, MODE, FV>(a, inj, tile, L.v);
    } else {
      stress_block<T, S, MODE, FS>(a, inj, tile, L.s);
    }
  } else record_point(rec, (int64_t)(bid - 2 * nb) * tile_threads(S) + threadIdx.y * WAVE + threadIdx.x);
}

// The injection by itself: lists too long or too spread for a step's blocks.
template <typename T, bool ACC, bool GRAD = false, bool PM = false>
__global__ void __launch_bounds__(256) k_inject(PointArgs<T> a) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= a.off[9]) return;
  const int c = comp_of(a, g);
  const int64_t k = g - a.off[c];
  if (a.pos[c][k] >= 0) inject_point<T, ACC, GRAD, PM>(a, c, k);
}

template <typename T>
__global__ void __launch_bounds__(256) k_record(PointArgs<T> a) {
  record_point(a, (int64_t)blockIdx.x * blockDim.x + threadIdx.x);
}

// Caller traces tr[c] = [n[c]][nts] of the 9 components <-> the time-major
// buffer tm = [nts][tot], component c at column off[c]. blockIdx.z = c.
template <typename T>
struct TransposeArgs {
  T* tr[9];
  T* tm;
  int64_t n[9], off[9];
  int64_t nts, tot;
};

template <typename T, bool TO_TM>
__global__ void __launch_bounds__(256) k_transpose(TransposeArgs<T> a) {
  __shared__ T tile[32][33];
  const int c = blockIdx.z;
  const int64_t p0 = (int64_t)blockIdx.x * 32, n = a.n[c];
  if (p0 >= n) return;  // block-uniform
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int64_t t0 = (int64_t)blockIdx.y * 32; t0 < a.nts; t0 += (int64_t)gridDim.y * 32) {
    for (int j = ty; j < 32; j += 8) {
      if (TO_TM ? (p0 + j < n && t0 + tx < a.nts) : (t0 + j < a.nts && p0 + tx < n))
        tile[j][tx] = TO_TM ? a.tr[c][(p0 + j) * a.nts + t0 + tx] : a.tm[(t0 + j) * a.tot + a.off[c] + p0 + tx];
    }
    __syncthreads();
    for (int j = ty; j < 32; j += 8) {
      if (TO_TM) {
        if (t0 + j < a.nts && p0 + tx < n) a.tm[(t0 + j) * a.tot + a.off[c] + p0 + tx] = tile[tx][j];
      } else if (p0 + j < n && t0 + tx < a.nts) {
        a.tr[c][(p0 + j) * a.nts + t0 + tx] = tile[tx][j];
      }
    }
    __syncthreads();
  }
}

// The 9 trace arrays cleared (blockIdx.y = component).
template <typename T>
__global__ void __launch_bounds__(256) k_clear_traces(TransposeArgs<T> a) {
  const int c = blockIdx.y;
  const int64_t n = a.n[c] * a.nts;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    a.tr[c][i] = T(0);
}

// Born forward secondary sources for coarse sample `its`
// (imagingElaFwdGpu_3D, kernelsElaGpu_3D.cu:1232-1438). V* are the coarse
// vx, vy, vz slices at its-1 (o), its (c), its+1 (n); o/n null at the ends.
template <typename T>
struct ImagingArgs {
  const T* o[3];
  const T* c[3];
  const T* n[3];
  const T* dm[8];   // scaled perturbations (drhox drhoy drhoz dlame dmu dmuxz dmuxy dmuyz)
  double* dmo[8];   // adjoint: accumulated images (FP64: summed over every coarse sample)
  T* ss[9];         // forward: secondary sources out; adjoint: adjoint coarse slices in
  T cx[4], cy[4], cz[4];
  T dts_inv;
  int its, nts;
  int init;         // adjoint: the images hold nothing yet (written, not read)
  int physics;      // 0: the yz term with the xz derivative pattern (reference); 1: the yz pattern
  int nz, nx, ny, nzi, zoff;
  int64_t ys;
  int ychunk, nbz, nbx, nby;
  int remap, xgroup;
  const int* chunks;
};

// The imaging kernels' LDS: double-buffered planes of the coarse vx, vy, vz
// slice V[its] (one LDS object, see k_step).
template <typename T, int S>
struct ImagingLds {
  Plane<T, S> vx[2], vy[2], vz[2];
};

// Secondary sources (forward) or images (adjoint) of coarse sample its. The
// strain rates of V[its] are those of the stress update (the same D+ / D-
// pattern), so the kernel runs the stress stepper's pipeline: planes of
// V[its] with x / z halos double-buffered in LDS (FP32 rows straight from
// HBM), y derivatives from 8-deep register queues, the next plane's loads
// issued before the current plane is computed, one barrier per plane, 32-bit
// offsets and unpredicated neighbour loads (every library array carries the
// guard that keeps them inside its allocation). Per interior cell it reads
// V[its - 1] and V[its + 1] (not at the ends of the record) and the 8
// perturbations (forward, writing 9 secondary sources) or the 9 adjoint
// slices and the 8 FP64 images (adjoint, rewriting the images).
template <typename T, int S, bool ADJ>
__global__ void __launch_bounds__(tile_threads(S)) k_imaging(ImagingArgs<T> a) {
  constexpr int BX = tile_x(S);
  __shared__ ImagingLds<T, S> L;
  auto& l_vx = L.vx; auto& l_vy = L.vy; auto& l_vz = L.vz;
  const TileCoord t = tile_coord<S>(blockIdx.x, a.nbz, a.nbx, a.nby, a.ychunk, a.nz, a.nzi, a.zoff, a.nx, a.ny, a.remap, a.xgroup, a.chunks);
  if (t.empty) return;  // block-uniform, before any barrier
  const uint32_t ys = (uint32_t)a.ys;
  constexpr bool DMA = ELA_LDS_DMA && sizeof(T) == 4;
  const int r = t.ty + FAT, q = t.tz + FAT;
  const int wy = __builtin_amdgcn_readfirstlane(t.ty), wr = wy + FAT;  // wave-uniform row
  const bool first = a.its == 0, last = a.its == a.nts - 1;            // kernel-uniform

  struct Stage {
    T hlo[3], hhi[3], hz[3];   // x-halo rows and z-halo column of vx, vy, vz
    T nx, ny, nz;              // new queue values (vx: plane + 3, vy: + 4, vz: + 3)
  };
  auto fetch = [&](Stage& v, int p, int nb) {
    const uint32_t pl = (uint32_t)p * ys;
    v.nx = *at(a.c[0], pl + 3 * ys + t.col);
    v.ny = *at(a.c[1], pl + 4 * ys + t.col);
    v.nz = *at(a.c[2], pl + 3 * ys + t.col);
    if (wy < FAT) {  // the x-halo loaders are whole waves
      if constexpr (DMA) {
        rows_to_lds<S>(a.c[0], pl + t.cxl, l_vx[nb], wy, FAT); rows_to_lds<S>(a.c[0], pl + t.cxh, l_vx[nb], wr + BX, FAT);
        rows_to_lds<S>(a.c[1], pl + t.cxl, l_vy[nb], wy, FAT); rows_to_lds<S>(a.c[1], pl + t.cxh, l_vy[nb], wr + BX, FAT);
        rows_to_lds<S>(a.c[2], pl + t.cxl, l_vz[nb], wy, FAT); rows_to_lds<S>(a.c[2], pl + t.cxh, l_vz[nb], wr + BX, FAT);
      } else {
#pragma unroll
        for (int f = 0; f < 3; ++f) { v.hlo[f] = *at(a.c[f], pl + t.cxl); v.hhi[f] = *at(a.c[f], pl + t.cxh); }
      }
    }
    if (t.zh) {
#pragma unroll
      for (int f = 0; f < 3; ++f) v.hz[f] = *at(a.c[f], pl + t.czh);
    }
  };
  auto stage = [&](int b, const Stage& v, T cvx, T cvy, T cvz) {
    l_vx[b][r][q] = cvx; l_vy[b][r][q] = cvy; l_vz[b][r][q] = cvz;
    if (!DMA && t.xh) {
      l_vx[b][t.ty][q] = v.hlo[0]; l_vx[b][r + BX][q] = v.hhi[0];
      l_vy[b][t.ty][q] = v.hlo[1]; l_vy[b][r + BX][q] = v.hhi[1];
      l_vz[b][t.ty][q] = v.hlo[2]; l_vz[b][r + BX][q] = v.hhi[2];
    }
    if (t.zh) { l_vx[b][r][t.colh] = v.hz[0]; l_vy[b][r][t.colh] = v.hz[1]; l_vz[b][r][t.colh] = v.hz[2]; }
  };

  // queues: vx (D-y, q[j] = f[iy-4+j]), vy (D+y, f[iy-3+j]), vz (D-y)
  T qx[8], qy[8], qz[8];
#pragma unroll
  for (int j = 0; j < 7; ++j) {
    qx[j] = *at(a.c[0], (uint32_t)(t.y0 - 4 + j) * ys + t.col);
    qy[j] = *at(a.c[1], (uint32_t)(t.y0 - 3 + j) * ys + t.col);
    qz[j] = *at(a.c[2], (uint32_t)(t.y0 - 4 + j) * ys + t.col);
  }
  {
    Stage v0;
    fetch(v0, t.y0, 0);
    qx[7] = v0.nx; qy[7] = v0.ny; qz[7] = v0.nz;
    stage(0, v0, qx[4], qy[3], qz[4]);
  }
  __syncthreads();
  int b = 0;
  for (int iy = t.y0; iy < t.y1; ++iy) {
    const bool more = iy + 1 < t.y1;
    Stage nx_;
    if (more) fetch(nx_, iy + 1, b ^ 1);  // buffer b ^ 1 is free: every wave passed the last barrier
    if (t.active) {
      const uint32_t i = (uint32_t)iy * ys + t.col;
      // every per-cell operand is loaded before the first store (a load
      // behind a store that might alias it waits for that store)
      T dv[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const T o = first ? T(0) : *at(a.o[k], i);
        const T n = last ? T(0) : *at(a.n[k], i);
        dv[k] = o - n;   // V[its-1] - V[its+1], zero outside the record
      }
      T dm[8], ss[9];
      double dmo[8];
      if constexpr (!ADJ) {
#pragma unroll
        for (int k = 0; k < 8; ++k) dm[k] = *at(a.dm[k], i);
      } else {
#pragma unroll
        for (int k = 0; k < 9; ++k) ss[k] = *at(a.ss[k], i);
#pragma unroll
        for (int k = 0; k < 8; ++k) dmo[k] = a.init ? 0.0 : a.dmo[k][i];   // 64-bit indexing: FP64 offsets can pass 4 GiB
      }
      const T* cx = a.cx; const T* cy = a.cy; const T* cz = a.cz;
      const T exx = dpx<T, S>(l_vx[b], r, q, cx);
      const T eyy = dq(qy, cy);
      const T ezz = dpz<T, S>(l_vz[b], r, q, cz);
      const T gxy = dq(qx, cy) + dmx<T, S>(l_vy[b], r, q, cx);
      const T gxz = dmz<T, S>(l_vx[b], r, q, cz) + dmx<T, S>(l_vz[b], r, q, cx);
      // yz term: the reference uses the xz derivative pattern
      // (kernelsElaGpu_3D.cu:1419-1431, :1622-1634); physics mode the yz one
      // of the stepper's syz update (D-y vz + D-z vy)
      const T gyz = a.physics ? dq(qz, cy) + dmz<T, S>(l_vy[b], r, q, cz) : gxz;
      if constexpr (!ADJ) {
#pragma unroll
        for (int k = 0; k < 3; ++k) st_nt(a.ss[k], i, dm[k] * dv[k] * a.dts_inv);
        const T div = exx + eyy + ezz;
        st_nt(a.ss[SXX], i, dm[3] * div + T(2.0) * dm[4] * exx);
        st_nt(a.ss[SYY], i, dm[3] * div + T(2.0) * dm[4] * eyy);
        st_nt(a.ss[SZZ], i, dm[3] * div + T(2.0) * dm[4] * ezz);
        st_nt(a.ss[SXZ], i, dm[5] * gxz);
        st_nt(a.ss[SXY], i, dm[6] * gxy);
        st_nt(a.ss[SYZ], i, dm[7] * gyz);
      } else {
        // each coarse sample's term in T, the sum over samples in FP64
#pragma unroll
        for (int k = 0; k < 3; ++k) a.dmo[k][i] = dmo[k] + double(ss[k] * dv[k] * a.dts_inv);
        const T sxx = ss[SXX], syy = ss[SYY], szz = ss[SZZ];
        a.dmo[3][i] = dmo[3] + double((sxx + syy + szz) * (exx + eyy + ezz));
        a.dmo[4][i] = dmo[4] + double(T(2.0) * (exx * sxx + eyy * syy + ezz * szz));
        a.dmo[5][i] = dmo[5] + double(ss[SXZ] * gxz);
        a.dmo[6][i] = dmo[6] + double(ss[SXY] * gxy);
        a.dmo[7][i] = dmo[7] + double(ss[SYZ] * gyz);
      }
    }
#pragma unroll
    for (int j = 0; j < 7; ++j) { qx[j] = qx[j + 1]; qy[j] = qy[j + 1]; qz[j] = qz[j + 1]; }
    if (more) {
      qx[7] = nx_.nx; qy[7] = nx_.ny; qz[7] = nx_.nz;
      stage(b ^ 1, nx_, qx[4], qy[3], qz[4]);
    }
    __syncthreads();
    b ^= 1;
  }
}

// Reference-layout flat indices -> internal-layout offsets. Positions outside
// the FD interior are replaced by -1 (skipped by the point kernels) and
// reported through *bad; box (or null) becomes the box of the others (see
// inject_tile).
struct ConvertArgs {
  const int64_t* in[14];   // 7 source lists, 7 receiver lists
  int64_t off[15];         // prefix offsets over the lists
  int32_t* out;            // the converted lists, one after another
  int nz, nx, ny, nzi, zoff;
  const int* ytab;
  int* bad;
  int* box[2];             // of the sources and of the receivers, or null
};

__global__ void __launch_bounds__(256) k_convert_pos(ConvertArgs a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.off[14]) return;
  int l = 0;
#pragma unroll
  for (int k = 1; k < 14; ++k) l += i >= a.off[k] ? 1 : 0;
  const int64_t p = a.in[l][i - a.off[l]];
  const int nz = a.nz, nx = a.nx, ny = a.ny;
  const int64_t ys = (int64_t)nz * nx;
  const int64_t iy = (p >= 0 && p < ys * ny) ? p / ys : -1;
  const int64_t r = p - iy * ys;
  const int64_t ix = r / nz, iz = r - ix * nz;
  bool ok = iy >= FAT && iy < ny - FAT && ix >= FAT && ix < nx - FAT && iz >= FAT && iz < nz - FAT;
  if (ok && a.ytab) {  // inside the interior of its window
    const int wy0 = a.ytab[4 * iy], wny = a.ytab[4 * iy + 1], wnx = a.ytab[4 * iy + 2];
    ok = wny > 0 && iy >= wy0 + FAT && iy < wy0 + wny - FAT && ix < wnx - FAT;
  }
  a.out[i] = ok ? (int32_t)(iy * nx * a.nzi + ix * a.nzi + iz + a.zoff) : -1;
  int* box = a.box[l >= 7];
  if (!ok) atomicOr(a.bad, 1);
  else if (box) {
    const int c[3] = {(int)iz + a.zoff, (int)ix, (int)iy};
    for (int k = 0; k < 3; ++k) { atomicMax(box + 2 * k, POS_TOP - c[k]); atomicMax(box + 2 * k + 1, c[k]); }
  }
}

// Device-side coarse-step counter of a replayed graph: *c += delta.
__global__ void k_count(int* c, int delta) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *c += delta;
}

template <typename T>
__global__ void __launch_bounds__(256) k_fill(T* p, int64_t n, T v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = i; k < n; k += stride) p[k] = v;
}

// ---------------------------------------------------------------------------
// Checkpoints of the forward state for the adjoint-state gradient: the 18
// arrays (two time levels x 9 fields) packed to the FD interior, either as
// they are or in bfloat16 scaled per array and per snapshot by a power of two
// 2^e >= max |x| (the scaling is exact; bfloat16 keeps 8 significant bits,
// rounded to nearest even).
// ---------------------------------------------------------------------------
// Unsigned 32-bit division by an invariant divisor d with a multiply-high,
// a subtraction and two shifts (Granlund and Montgomery, "Division by
// invariant integers using multiplication", PLDI 1994, section 4): with
// l = ceil(log2 d) and m = floor(2^32 (2^l - d) / d) + 1, t = mulhi(m, n),
// n / d = (t + ((n - t) >> min(l, 1))) >> max(l - 1, 0) for every 32-bit n.
// The host forms (m, l) once per grid (fast_div); the device avoids the
// 30-odd instructions of a general 32-bit division per element.
struct FastDiv {
  uint32_t m;
  int s1, s2;
};

__device__ __forceinline__ uint32_t fdiv(uint32_t n, FastDiv f) {
  const uint32_t t = __umulhi(f.m, n);
  return (t + ((n - t) >> f.s1)) >> f.s2;
}

template <typename T>
struct CkArgs {
  T* f[18];
  int nzI, nxI, nyI;     // interior extents (n - 2 FAT)
  int nzi, zoff;         // internal row pitch and z origin
  int64_t ys;            // nx * nzi
  int64_t nI;            // nzI * nxI * nyI
  FastDiv dz, dx;        // division by nzI and nxI
};

// Library offset of packed interior index q (32-bit: nI and every offset fit
// in 32 bits, the arrays being smaller than 4 GiB).
template <typename T>
__device__ __forceinline__ int64_t ck_offset(const CkArgs<T>& a, int64_t q) {
  const uint32_t q32 = (uint32_t)q, nz = (uint32_t)a.nzI, nx = (uint32_t)a.nxI;
  const uint32_t r = fdiv(q32, a.dz), iz = q32 - r * nz;
  const uint32_t iy = fdiv(r, a.dx), ix = r - iy * nx;
  return (int64_t)((iy + FAT) * (uint32_t)a.ys + (ix + FAT) * (uint32_t)a.nzi + (uint32_t)(a.zoff + FAT) + iz);
}

// Whether an interior cell of the grid lies in the interior of a window
// (ytab: per plane {window y0, ny, nx, window}, zeros between the windows).
__device__ __forceinline__ bool in_window(const int* ytab, int ix, int iy) {
  const int wy0 = ytab[4 * iy], wny = ytab[4 * iy + 1], wnx = ytab[4 * iy + 2];
  return iy >= wy0 + FAT && iy < wy0 + wny - FAT && ix < wnx - FAT;
}

__device__ __forceinline__ uint16_t f32_to_bf16(float x) {
  uint32_t u = __float_as_uint(x);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// Power-of-two scale >= amax (1 for an all-zero array).
__device__ __forceinline__ float pow2_scale(uint32_t amax_bits) {
  const float m = __uint_as_float(amax_bits);
  if (!(m > 0.f)) return 1.f;
  int e;
  const float fr = frexpf(m, &e);  // m = fr * 2^e, fr in [0.5, 1)
  (void)fr;
  return ldexpf(1.f, e);
}

// amax[f] = max |x| over the interior of array f (blockIdx.y = f), as the bit
// pattern of a non-negative float (ordered like unsigned integers).
template <typename T>
__global__ void __launch_bounds__(256) k_ck_amax(CkArgs<T> a, uint32_t* amax) {
  __shared__ float red[256];
  const int f = blockIdx.y;
  float m = 0.f;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < a.nI; q += (int64_t)gridDim.x * blockDim.x)
    m = fmaxf(m, fabsf((float)a.f[f][ck_offset(a, q)]));
  red[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicMax(&amax[f], __float_as_uint(red[0]));
}

// Pack: out[f][q] = x / scale_f as bfloat16 (BF16 = true) or x (BF16 = false).
template <typename T, bool BF16>
__global__ void __launch_bounds__(256) k_ck_pack(CkArgs<T> a, void* out, const uint32_t* amax, float* scale) {
  const int f = blockIdx.y;
  const float s = BF16 ? pow2_scale(amax[f]) : 1.f;
  const float inv = 1.f / s;   // exact: s is a power of two
  if (BF16 && blockIdx.x == 0 && threadIdx.x == 0) scale[f] = s;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < a.nI; q += (int64_t)gridDim.x * blockDim.x) {
    const T x = a.f[f][ck_offset(a, q)];
    if (BF16) static_cast<uint16_t*>(out)[f * a.nI + q] = f32_to_bf16((float)x * inv);
    else static_cast<T*>(out)[f * a.nI + q] = x;
  }
}

template <typename T, bool BF16>
__global__ void __launch_bounds__(256) k_ck_unpack(CkArgs<T> a, const void* in, const float* scale) {
  const int f = blockIdx.y;
  const float s = BF16 ? scale[f] : 1.f;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < a.nI; q += (int64_t)gridDim.x * blockDim.x) {
    T x;
    if (BF16) x = (T)(bf16_to_f32(static_cast<const uint16_t*>(in)[f * a.nI + q]) * s);
    else x = static_cast<const T*>(in)[f * a.nI + q];
    a.f[f][ck_offset(a, q)] = x;
  }
}

// The 8 scaled medium arrays from (rho, lambda, mu) on every cell of the
// padded grid with the host scaling's edge rules (the half-cell average
// halves the first sample and adds half the neighbour to the last one): the
// device twin of ela_scale_medium, same operations in the same order (FP32
// buoyancies and normal moduli formed in FP64 as in the steppers: buoy_h,
// normal_moduli).
template <typename T>
struct MedArgs {
  const T* ep[3];        // rho, lambda, mu (internal layout)
  T* m[8];               // the 8 scaled arrays (internal layout)
  int nz, nx, ny, nzi, zoff;
  int64_t ys;
  T tdt;
  double tdt64;
};

template <typename T>
__device__ __forceinline__ T half_cell(const T* f, int64_t i, int64_t s, int ia, int n) {
  return ia == 0 ? T(0.5) * f[i] : (ia < n - 1 ? T(0.5) * (f[i] + f[i - s]) : f[i] + T(0.5) * f[i - s]);
}
// the same in FP64 from the array's values (the FP32 buoyancies)
template <typename T>
__device__ __forceinline__ double half_cell64(const T* f, int64_t i, int64_t s, int ia, int n) {
  const double c = double(f[i]);
  return ia == 0 ? 0.5 * c : (ia < n - 1 ? 0.5 * (c + double(f[i - s])) : c + 0.5 * double(f[i - s]));
}

template <typename T>
__global__ void __launch_bounds__(256) k_scale_medium(MedArgs<T> a) {
  const int64_t n = (int64_t)a.nz * a.nx * a.ny;
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n; c += (int64_t)gridDim.x * blockDim.x) {
    const int iz = (int)(c % a.nz);
    const int64_t rest = c / a.nz;
    const int ix = (int)(rest % a.nx), iy = (int)(rest / a.nx);
    const int64_t i = iy * a.ys + (int64_t)ix * a.nzi + a.zoff + iz;
    const int64_t sx = a.nzi, sy = a.ys;
    const T* rho = a.ep[0];
    const T* lam = a.ep[1];
    const T* mu = a.ep[2];
    if constexpr (sizeof(T) == 4) {
      a.m[BX_][i] = buoy_h<T>(a.tdt, a.tdt64, half_cell64(rho, i, sx, ix, a.nx));
      a.m[BY_][i] = buoy_h<T>(a.tdt, a.tdt64, half_cell64(rho, i, sy, iy, a.ny));
      a.m[BZ_][i] = buoy_h<T>(a.tdt, a.tdt64, half_cell64(rho, i, (int64_t)1, iz, a.nz));
    } else {
      a.m[BX_][i] = a.tdt / half_cell(rho, i, sx, ix, a.nx);
      a.m[BY_][i] = a.tdt / half_cell(rho, i, sy, iy, a.ny);
      a.m[BZ_][i] = a.tdt / half_cell(rho, i, (int64_t)1, iz, a.nz);
    }
    normal_moduli(a.tdt, a.tdt64, lam[i], mu[i], a.m[L2M][i], a.m[LAM][i]);
    // mu staggered along x, then along z (muxz) or y (muxy); along y, then z (muyz)
    const T tx = half_cell(mu, i, sx, ix, a.nx);
    const T tx_z = iz > 0 ? half_cell(mu, i - 1, sx, ix, a.nx) : T(0);
    const T tx_y = iy > 0 ? half_cell(mu, i - sy, sx, ix, a.nx) : T(0);
    const T ty = half_cell(mu, i, sy, iy, a.ny);
    const T ty_z = iz > 0 ? half_cell(mu, i - 1, sy, iy, a.ny) : T(0);
    auto outer = [](T v, T vm, int ia, int na) {
      return ia == 0 ? T(0.5) * v : (ia < na - 1 ? T(0.5) * (v + vm) : v + T(0.5) * vm);
    };
    a.m[MXZ][i] = outer(tx, tx_z, iz, a.nz) * a.tdt;
    a.m[MXY][i] = outer(tx, tx_y, iy, a.ny) * a.tdt;
    a.m[MYZ][i] = outer(ty, ty_z, iz, a.nz) * a.tdt;
  }
}

// fluid[w] = 1 if the buoyancies or shear moduli of any interior cell of window
// w (without ytab: of the grid, w = 0) are not safely divided by (see
// check_solid). NaN counts as such. At most one atomic a wave and window.
template <typename T>
__global__ void __launch_bounds__(256) k_check_solid(CkArgs<T> a, const int* ytab, int* fluid) {
  int told = -1;   // the last window this lane's wave has reported
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < a.nI; q += (int64_t)gridDim.x * blockDim.x) {
    int w = 0;
    if (ytab) {
      const uint32_t r = fdiv((uint32_t)q, a.dz), iy = fdiv(r, a.dx), ix = r - iy * (uint32_t)a.nxI;
      if (!in_window(ytab, (int)ix + FAT, (int)iy + FAT)) continue;
      w = ytab[4 * (iy + FAT) + 3];
    }
    const int64_t i = ck_offset(a, q);
    constexpr T tiny = T(0x1p-64);
    const T least = max(a.f[L2M][i] * T(0x1p-20), tiny);
    bool ok = a.f[L2M][i] > T(0);
    for (int k = MXZ; k <= MYZ; ++k) ok = ok && a.f[k][i] >= least;
    for (int k = BX_; k <= BZ_; ++k) ok = ok && a.f[k][i] >= tiny;
    if (!ok && w != told) {
      told = w;
      const int first = __ffsll((unsigned long long)__ballot(1)) - 1;
      if ((int)(threadIdx.x & 63) == first || w != __builtin_amdgcn_readfirstlane(w)) atomicOr(fluid + w, 1);
    }
  }
}

// Streaming reference for the roofline: R arrays of n4 16-byte vectors are
// read and the first W of them rewritten in place (non-temporal stores), the
// byte mix of a stencil kernel (reads of c, o and the medium, o rewritten)
// without neighbour accesses. Grid-stride loop over vectors. W = 0 reads
// only: the sum of all four lanes of the vector sum is compared with a value
// the (zero-filled) inputs never give, so every load stays live and nothing
// is written.
template <int R, int W>
__global__ void __launch_bounds__(256) k_stream(float4* const* arrays, int64_t n4) {
  float4* a[R];
#pragma unroll
  for (int k = 0; k < R; ++k) a[k] = arrays[k];
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (int64_t)gridDim.x * blockDim.x) {
    float4 s = a[0][i];
#pragma unroll
    for (int k = 1; k < R; ++k) {
      const float4 v = a[k][i];
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    if constexpr (W == 0) {
      if (s.x + s.y + s.z + s.w == -1.2345e30f) a[0][i] = s;
    }
#pragma unroll
    for (int k = 0; k < W; ++k) {
      typedef float f4 __attribute__((ext_vector_type(4)));
      const f4 o = {s.x + (float)k, s.y, s.z, s.w};
      __builtin_nontemporal_store(o, reinterpret_cast<f4*>(a[k] + i));
    }
  }
}

// 16-bit checkpoints with one scale per block of CK_BLOCK consecutive packed
// values: q = rint(x / s) with s = max |x| / 32767 over the block (an
// all-zero block has s = 0), restored as x = q s. The absolute error is at
// most s / 2 (2^-16 of the block's largest value), against 2^-9 of each value
// for bfloat16. Layout of one checkpoint: int16 [18][nI], then float scales
// [18][ceil(nI / CK_BLOCK)] (36 nI bytes precede them, so they are 4-byte
// aligned). One wave quantises one block (the max is a wave reduction).
constexpr int CK_BLOCK = 64;

template <typename T>
__global__ void __launch_bounds__(256) k_ck_pack_s16(CkArgs<T> a, int16_t* out) {
  const int f = blockIdx.y;
  const int64_t nb = (a.nI + CK_BLOCK - 1) / CK_BLOCK;
  int16_t* q16 = out + f * a.nI;
  float* sc = reinterpret_cast<float*>(out + 18 * a.nI) + f * nb;
  const int lane = threadIdx.x & (CK_BLOCK - 1);
  const int64_t wstride = (int64_t)gridDim.x * (blockDim.x / CK_BLOCK);
  // b is uniform over a wave (blockDim.x is a multiple of 64), so every lane joins the reduction:
  // the maximum of each 32-lane half (DPP row moves and a swizzle), then of the two halves
  for (int64_t b = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / CK_BLOCK; b < nb; b += wstride) {
    const int64_t q = b * CK_BLOCK + lane;
    const bool ok = q < a.nI;
    const float x = ok ? (float)a.f[f][ck_offset(a, q)] : 0.f;
    const float h = half_wave_absmax(x);
    const float m = fmaxf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(h), 0)),
                          __int_as_float(__builtin_amdgcn_readlane(__float_as_int(h), 32)));
    const float inv = m > 0.f ? 32767.f / m : 0.f;
    if (ok) q16[q] = (int16_t)__float2int_rn(x * inv);
    if (lane == 0) sc[b] = m / 32767.f;
  }
}

template <typename T>
__global__ void __launch_bounds__(256) k_ck_unpack_s16(CkArgs<T> a, const int16_t* in) {
  const int f = blockIdx.y;
  const int64_t nb = (a.nI + CK_BLOCK - 1) / CK_BLOCK;
  const int16_t* q16 = in + f * a.nI;
  const float* sc = reinterpret_cast<const float*>(in + 18 * a.nI) + f * nb;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < a.nI; q += (int64_t)gridDim.x * blockDim.x)
    a.f[f][ck_offset(a, q)] = (T)((float)q16[q] * sc[q / CK_BLOCK]);
}

// Vectorised k_ck_pack_s16 / k_ck_unpack_s16 for FP32 grids whose interior
// z extent is a multiple of 8 (so are nI and every row start): a lane moves 8
// consecutive values -- 32 bytes of one z row (two 16-byte loads or stores)
// and 16 bytes of the packed int16 -- instead of one 4-byte and one 2-byte
// access, which kept too few bytes in flight per lane to reach the HBM rate.
// The 8 lanes of a 64-value block form its maximum with DPP moves inside
// their 8-lane group. Same blocks, scales and values as the scalar kernels.
__global__ void __launch_bounds__(256) k_ck_pack_s16_v8(CkArgs<float> a, int16_t* out) {
  const int f = blockIdx.y;
  const int64_t nb = (a.nI + CK_BLOCK - 1) / CK_BLOCK, n8 = a.nI / 8;
  int16_t* q16 = out + f * a.nI;
  float* sc = reinterpret_cast<float*>(out + 18 * a.nI) + f * nb;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  // g0 is uniform over the block, so every lane joins the reductions (lanes past the end hold zeros)
  for (int64_t g0 = (int64_t)blockIdx.x * blockDim.x; g0 < n8; g0 += stride) {
    const int64_t g = g0 + threadIdx.x;
    const bool ok = g < n8;
    float4 u = make_float4(0.f, 0.f, 0.f, 0.f), v = u;
    if (ok) {
      const float4* p = reinterpret_cast<const float4*>(a.f[f] + ck_offset(a, g * 8));
      u = p[0];
      v = p[1];
    }
    const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
    uint32_t mu = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) mu = max(mu, __float_as_uint(fabsf(x[k])));
    mu = dpp_umax<0xB1>(mu);   // quad_perm [1, 0, 3, 2]
    mu = dpp_umax<0x4E>(mu);   // quad_perm [2, 3, 0, 1]
    mu = dpp_umax<0x141>(mu);  // row_half_mirror: the 8-lane group's maximum
    const float m = __uint_as_float(mu);
    const float inv = m > 0.f ? 32767.f / m : 0.f;
    if (ok) {
      uint32_t w[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        w[k] = (uint32_t)(uint16_t)(int16_t)__float2int_rn(x[2 * k] * inv) |
               ((uint32_t)(uint16_t)(int16_t)__float2int_rn(x[2 * k + 1] * inv) << 16);
      *reinterpret_cast<uint4*>(q16 + g * 8) = make_uint4(w[0], w[1], w[2], w[3]);
      if ((threadIdx.x & 7) == 0) sc[g / 8] = m / 32767.f;
    }
  }
}

__global__ void __launch_bounds__(256) k_ck_unpack_s16_v8(CkArgs<float> a, const int16_t* in) {
  const int f = blockIdx.y;
  const int64_t nb = (a.nI + CK_BLOCK - 1) / CK_BLOCK, n8 = a.nI / 8;
  const int16_t* q16 = in + f * a.nI;
  const float* sc = reinterpret_cast<const float*>(in + 18 * a.nI) + f * nb;
  for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < n8; g += (int64_t)gridDim.x * blockDim.x) {
    const uint4 w = *reinterpret_cast<const uint4*>(q16 + g * 8);
    const float s = sc[g / 8];
    auto lo = [&](uint32_t b) { return (float)(int16_t)(uint16_t)(b & 0xFFFFu) * s; };
    auto hi = [&](uint32_t b) { return (float)(int16_t)(uint16_t)(b >> 16) * s; };
    float4* p = reinterpret_cast<float4*>(a.f[f] + ck_offset(a, g * 8));
    p[0] = make_float4(lo(w.x), hi(w.x), lo(w.y), hi(w.y));
    p[1] = make_float4(lo(w.z), hi(w.z), lo(w.w), hi(w.w));
  }
}

// The gradient's FP32 partial sums folded into its FP64 sums over the FD
// interior only (the steppers and injections write nothing else): four
// consecutive z values per lane (interior z extent a multiple of 4, rows
// 16-byte aligned), array m = blockIdx.y of a.f (partial sums) and of acc
// (FP64 sums, stride np); the partial sums are cleared. FIRST: the FP64 sums
// hold nothing yet (written, not read).
template <bool FIRST>
__global__ void __launch_bounds__(256) k_fold_v4(CkArgs<float> a, double* acc, int64_t np) {
  const int m = blockIdx.y;
  float* part = a.f[m];
  double* ac = acc + m * np;
  const int64_t n4 = a.nI / 4;
  for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < n4; g += (int64_t)gridDim.x * blockDim.x) {
    const int64_t o = ck_offset(a, g * 4);
    float4* pp = reinterpret_cast<float4*>(part + o);
    double2* d = reinterpret_cast<double2*>(ac + o);
    const float4 p = *pp;
    double2 d0 = make_double2(0.0, 0.0), d1 = d0;
    if constexpr (!FIRST) { d0 = d[0]; d1 = d[1]; }
    d0.x += (double)p.x; d0.y += (double)p.y;
    d1.x += (double)p.z; d1.y += (double)p.w;
    d[0] = d0;
    d[1] = d1;
    *pp = make_float4(0.f, 0.f, 0.f, 0.f);
  }
}

// acc[i] (+)= (double) part[i]; part[i] = 0 over whole arrays.
template <typename T, bool FIRST>
__global__ void __launch_bounds__(256) k_fold(T* part, double* acc, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    acc[i] = (FIRST ? 0.0 : acc[i]) + (double)part[i];
    part[i] = T(0);
  }
}

// The sums of a call added to the caller's arrays [8][ny][nx][nz] over the FD
// interior (ytab: over the windows' interiors, the only cells whose sums the
// steps write), in place: out = U(double(out) + acc (+ part)), acc the FP64
// sums (stride np; null: part alone), part the gradient's last partial sums
// (null: none). Takes the place of copying the caller's arrays in, converting them,
// adding and copying them out: Born adjoint 232x328x324 (40 steps) 77.2 ->
// 75.5 ms, gradient 99.8 -> 98.3 ms.
template <typename T, typename U>
__global__ void __launch_bounds__(256) k_add_out(CkArgs<T> a, const double* acc, const T* part, int64_t np, U* out,
                                                 int nz, int nx, int64_t n_model, const int* ytab) {
  const int m = blockIdx.y;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < a.nI; q += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t q32 = (uint32_t)q, r = fdiv(q32, a.dz), iz = q32 - r * (uint32_t)a.nzI;
    const uint32_t iy = fdiv(r, a.dx), ix = r - iy * (uint32_t)a.nxI;
    if (ytab && !in_window(ytab, (int)ix + FAT, (int)iy + FAT)) continue;
    const int64_t i = (int64_t)((iy + FAT) * (uint32_t)a.ys + (ix + FAT) * (uint32_t)a.nzi + (uint32_t)(a.zoff + FAT) + iz);
    double s = acc ? acc[m * np + i] : 0.0;
    if (part) s += (double)part[m * np + i];
    U* o = out + m * n_model + ((int64_t)(iy + FAT) * nx + (ix + FAT)) * nz + FAT + iz;
    *o = U((double)*o + s);
  }
}

}  // namespace ela
