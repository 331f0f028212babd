// smc_tile.hip -- exact-footprint Gaussian smearing on VALU tiles.
//
// The smearing of MCnucl.cpp:432-478 (T_A / T_B), :689-760 (MC-Glauber
// entropy) and :762-811 (sqrt(T_A T_B)) adds, for every source k inside its
// integer footprint window and inside the disk dx^2 + dy^2 <= 25 w^2
// (Particle.cpp:122-132),
//     T[x][y] += w_k gx_k(x) gy_k(y),   g(d) = exp(-d^2 / (2 w^2)).
//
// The disk cut without a compare.  Inside the disk gx gy >= theta =
// exp(-cut2 / (2 w^2)), outside it gx gy < theta.  The row factor is stored
// as K gx with K = 2^-126 / theta, so the product p = (K gx) gy is a normal
// float exactly when the cell is inside the disk and a denormal otherwise.
// This file is compiled with f32 denormals flushed (the kernel's MODE
// register flushes the outputs of v_mul_f32), so cells outside the disk
// get p = 0 and every cell costs one multiply and one FMA:
//     acc += p * (w_k 2^64),    T = acc * 2^-64 / K
// (2^64 keeps w_k p far above the denormal range for any w_k > 2^-64).
// The boundary is that of the product in float, within a few ulp of the
// exact disk.  Without a cut (cut2 = 1e30) K = 2^64, nothing flushes and
// the footprint is the integer window alone.
//
// One workgroup owns a tile of 32 rows x 64 columns of an event: one wave, or
// four or sixteen where a batch has too few tiles to fill the chip (a tile is
// a serial chain over its sources).  The sources of the list whose window
// meets the tile are selected in source order (ballot compaction, so every
// cell adds its terms in one fixed order whatever the shape) and taken a few
// at a time: row factors K gx and column factors gy go to LDS once per source,
// then each lane adds its cells.
//
// In the one-wave kernel lane (q, c) = (lane / 16, lane % 16) holds the cells of rows q + 4 i and
// columns c + 16 k: a source costs a lane TR / 4 row and 4 column factors, read
// as float4, for TR cells.  (With lane = column a cell needs its own row
// factor from LDS, and the LDS return path, 128 B per clock and CU, is as busy
// as the VALU: a layout with fewer VALU instructions then gained nothing.)
// Register (i, k) of a wave is a 4 x 16 patch, so a source's work is skipped in
// units of 16 x 16 cells that its window or its disk does not reach: 3,800 cell
// slots of 6,700 in 8-row chunks of 64 columns remain for a 51-cell window.  At the end the 4 x 4 blocks (q, k) are
// transposed across the lane groups, and a lane holds one column again:
// stores of 64 consecutive cells.
#include <algorithm>

#include "smc_device.h"

namespace smc {

// a selected source: position (half-quanta) and window per axis, weight, and
// the units of the wave's tile that it reaches (bit 4 row unit + column block)
struct alignas(8) TileEntry {
  int xh, xw;
  int yh, yw;
  float w;
  unsigned units;
};

constexpr int kTileRows = 32;  // rows of a workgroup's tile

// The 4 x 4 transpose of v over (lane group of 16, register):
// v[k] of group q <- v[q] of group k.
__device__ __forceinline__ void transpose_groups(float (&v)[4]) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const auto swap32 = [](float& a, float& b) {
    const u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r.x);
    b = __uint_as_float(r.y);
  };
  const auto swap16 = [](float& a, float& b) {
    const u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r.x);
    b = __uint_as_float(r.y);
  };
  swap32(v[0], v[2]);
  swap32(v[1], v[3]);
  swap16(v[0], v[1]);
  swap16(v[2], v[3]);
}

// The MC-KLN density of MCnucl::setDensity (which_mc_model 1,
// MCnucl.cpp:654-687) fused into the smearing: T_A and T_B accumulate in two
// register sets of one wave, and each cell's dN/dy is the sixPoint2dInterp
// (arsenal.cpp:33-54) of the table at (T_A/dT, T_B/dT) in FP64, from the same
// float T values the separate k_tile + k_kln_table pair reads back.
struct KlnTab {
  const double* table;  // tmax x tmax, row = T_A index
  int tmax;
  double dT;
};

__device__ __forceinline__ float kln_cell(float A, float B, const KlnTab& kt, bool& out_of_table) {
  const double di = (double)A / kt.dT, dj = (double)B / kt.dT;
  if (!(di >= 0 && di < kt.tmax - 2) || !(dj >= 0 && dj < kt.tmax - 2)) {  // also catches NaN
    out_of_table = true;
    return 0.f;
  }
  // row and column 0 of the table are 0, so T_A = 0 or T_B = 0 gives 0
  if (A == 0.f || B == 0.f) return 0.f;
  const int a = (int)floor(di), b = (int)floor(dj);
  const double x = di - a, y = dj - b;
  const double* t = kt.table;
  const int m = kt.tmax;
  const double v00 = t[a * m + b], v01 = t[a * m + b + 1], v02 = t[a * m + b + 2];
  const double v10 = t[(a + 1) * m + b], v11 = t[(a + 1) * m + b + 1];
  const double v20 = t[(a + 2) * m + b];
  const double axx = 1.0 / 2.0 * (v00 - 2 * v10 + v20);
  const double axy = v00 - v01 - v10 + v11;
  const double ayy = 1.0 / 2.0 * (v00 - 2 * v01 + v02);
  const double bx = 1.0 / 2.0 * (-3.0 * v00 + 4 * v10 - v20);
  const double by = 1.0 / 2.0 * (-3.0 * v00 + 4 * v01 - v02);
  return (float)(axx * x * x + axy * x * y + ayy * y * y + bx * x + by * y + v00);
}

// Event and tile of a workgroup.  Workgroups go to the 8 XCDs round-robin by
// linear id; this mapping gives all tiles of an event one XCD (one L2 holds
// its source list, and the partial cache lines at tile edges meet in that
// L2).  spread: the tiles of an event go to all XCDs instead (few events: one
// XCD has 32 CUs).
struct TileAt {
  int e, tile, T, R0, c0;  // e < 0: no event
  bool col_live;  // the event's source rectangle reaches the tile's columns
  int x0, x1;     // its rows
};
__device__ __forceinline__ TileAt tile_at(const DevCfg& cfg, const EvBufs& buf, int nev, int spread,
                                          const int* order) {
  const int ntx = (cfg.nx + kTileRows - 1) / kTileRows;
  TileAt at;
  at.T = ntx * ((cfg.ny + 63) >> 6);
  const unsigned L = blockIdx.x, rg = L % (8u * at.T);
  at.e = spread ? (int)(L / at.T) : (int)(8u * (L / (8u * at.T)) + rg % 8u);
  at.tile = spread ? (int)(L % at.T) : (int)(rg / 8u);
  at.R0 = kTileRows * (at.tile % ntx);
  at.c0 = 64 * (at.tile / ntx);
  at.e = at.e < nev ? (order ? order[at.e] : at.e) : -1;
  const int e = max(at.e, 0);
  const int rx = buf.counts[(size_t)e * 8 + 6], ry = buf.counts[(size_t)e * 8 + 7];
  at.col_live = (ry & 0xffff) < at.c0 + 64 && (ry >> 16) > at.c0;
  at.x0 = rx & 0xffff;
  at.x1 = rx >> 16;
  return at;
}

// The range of event e's source list that holds accumulator want's sources
// (the list is the projectile's participants, the target's, then the pairs).
__device__ __forceinline__ int2 source_range(const EvBufs& buf, const SmearSpec& spec, int e, int want) {
  const int* cnt = buf.counts + (size_t)e * 8;
  const int K = cnt[5];
  const int end[3] = {min(cnt[0], K), min(cnt[0] + cnt[1], K), K};
  int2 r = make_int2(K, 0);
#pragma unroll
  for (int kind = 0; kind < 3; ++kind)
    if (spec.enabled[kind] && spec.acc[kind] == want) {
      r.x = min(r.x, kind ? end[kind - 1] : 0);
      r.y = end[kind];
    }
  return r;
}

// The source (s, wv4) as an entry, with units != 0 if it belongs to
// accumulator want and reaches the rows r0 .. r0 + UROWS NU - 1 and columns
// c0 .. c0 + 63: bit 4 u + kb for rows [r0 + UROWS u, + UROWS), columns
// [c0 + 16 kb, + 16).  A unit is reached if the window meets it and its
// nearest cell lies within reach2: cut2 and a margin that covers the float
// product's own boundary (a few ulp of exp(-cut2 / 2w^2)).
template <int UROWS, int NU>
__device__ __forceinline__ TileEntry tile_entry(const DevCfg& cfg, const SmearSpec& spec, const int4& s,
                                                const int4& wv4, int want, int r0, int c0) {
  TileEntry en{0, 0, 0, 0, 0.f, 0u};
  const int kind = s.w;
  if (!(spec.enabled[kind] && spec.acc[kind] == want)) return en;
  en.xh = s.x;
  en.yh = s.y;
  en.xw = (spec.win[kind] == kWinBox) ? wv4.x : wv4.z;
  en.yw = (spec.win[kind] == kWinBox) ? wv4.y : wv4.w;
  en.w = spec.scale[kind] * (spec.use_fluct[kind] ? __int_as_float(s.z) : 1.f) * cfg.tile_w;
  const int xlo = en.xw & 0xffff, xhi = en.xw >> 16, ylo = en.yw & 0xffff, yhi = en.yw >> 16;
  if (!(xlo < r0 + UROWS * NU && xhi > r0 && ylo < c0 + 64 && yhi > c0)) return en;
  const float reach2 = cfg.cut2 * 1.001f;
  const float sx = (float)(en.xh * kH - cfg.xmin), sy = (float)(en.yh * kH - cfg.ymin);
  const float fdx = (float)cfg.dx, fdy = (float)cfg.dy;
  float d2y[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const int a = max(c0 + 16 * kb, ylo), b = min(c0 + 16 * kb + 16, yhi) - 1;
    const float d = fmaxf(0.f, fmaxf(a * fdy - sy, sy - b * fdy));
    d2y[kb] = a <= b ? d * d : 3.0e38f;
  }
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int a = max(r0 + UROWS * u, xlo), b = min(r0 + UROWS * (u + 1), xhi) - 1;
    const float d = fmaxf(0.f, fmaxf(a * fdx - sx, sx - b * fdx));
    if (a > b) continue;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      if (d * d + d2y[kb] <= reach2) en.units |= 1u << (4 * u + kb);
  }
  return en;
}

// EPI 1 (MC-KLN) and 2 (sqrt(T_A T_B), MCnucl.cpp:762-811): the sources of
// accumulator 0 (T_A), then those of accumulator 1 (T_B), each set in source
// order, and the output is the cell's dN/dy from the table, or
// sqrtf(T_A T_B) of the stored floats.  EPI 0: the sources of accumulator
// acc_sel only.
//
// What the kernels below do with the sums of rows r0 .. r0 + TR - 1 (lane =
// column; aA: T_A where there are two): the epilogue and the stores; the stored
// values are left in a.
template <int TR, int EPI>
__device__ __forceinline__ void tile_finish(const DevCfg& cfg, const EvBufs& buf, const TileAt& at, int r0, bool live,
                                            float (&a)[TR], const float (&aA)[EPI ? TR : 1], const KlnTab& kt,
                                            float* out) {
  constexpr bool TWO = EPI != 0;
  const int lane = threadIdx.x & 63, col = at.c0 + lane, nx = cfg.nx, ny = cfg.ny;
  const float so = cfg.tile_out;
  if constexpr (EPI == 2) {
    // sqrt(T_A T_B) of the stored floats; the product is formed in double,
    // so the result does not depend on the f32 denormal mode of this file
#pragma unroll
    for (int r = 0; r < TR; ++r) a[r] = (float)sqrt((double)(aA[r] * so) * (double)(a[r] * so));
  }
  if constexpr (EPI == 1) {  // dN/dy from (T_A, T_B) = (aA, a) as stored floats
    bool off = false;
#pragma unroll
    for (int r = 0; r < TR; ++r)
      a[r] = (live && col < ny && r0 + r < nx) ? kln_cell(aA[r] * so, a[r] * so, kt, off) : 0.f;
    if (off) atomicOr(&buf.counts[(size_t)at.e * 8 + 3], kStKlnTable);
  }
  const float os = TWO ? 1.f : so;  // stored value = a * os
  const size_t N = (size_t)nx * ny;
  float* o = out + (size_t)at.e * N + (size_t)r0 * ny + col;
#pragma unroll
  for (int r = 0; r < TR; ++r) {
    a[r] *= os;
    if (col < ny && r0 + r < nx) o[(size_t)r * ny] = a[r];
  }
}

// Adds the stored values of rows r0 .. r0 + TR - 1 to the column sums s0 =
// sum v and s1 = sum x v, in row order whatever the shape: the centre of mass
// is the same to the bit, and with it what is ill-conditioned in it (the
// order-1 angle of an averaged profile is one of rounding).
template <int TR>
__device__ __forceinline__ void column_sums(const DevCfg& cfg, const TileAt& at, int r0, const float (&a)[TR],
                                            double& s0, double& s1) {
  const int col = at.c0 + (threadIdx.x & 63);
#pragma unroll
  for (int r = 0; r < TR; ++r) {
    if (col < cfg.ny && r0 + r < cfg.nx) {
      const double v = (double)a[r];
      s0 += v;
      s1 = fma(cfg.xmin + (r0 + r) * cfg.dx, v, s1);
    }
  }
}

// A tile's centre-of-mass partials from its column sums s0 = sum v, s1 = sum x v
__device__ __forceinline__ void tile_cm(const DevCfg& cfg, const TileAt& at, double s0, double s1, double* cm_out) {
  const int lane = threadIdx.x & 63, col = at.c0 + lane;
  double s2 = (col < cfg.ny) ? (cfg.ymin + col * cfg.dy) * s0 : 0.0;
  s0 = wave_sum(s0);
  s1 = wave_sum(s1);
  s2 = wave_sum(s2);
  if (lane == 0) {
    double* p = cm_out + ((size_t)at.e * at.T + at.tile) * 4;
    p[0] = s0;
    p[1] = s1;
    p[2] = s2;
    p[3] = 0.0;
  }
}

// ---- one wave per tile, for batches that fill the chip: bound by VALU issue
// (0.276 instructions per SIMD and cycle, a chain of FMAs reaches 0.245; two
// instructions per cell slot, about 60 per source and tile around them).
// 4 sources' factors in LDS at a time and 72 VGPRs (7 waves per SIMD): 8.93 ms
// per 50,000 Pb+Pb events of 261^2 cells; 8 sources 9.45 (7 waves) and 9.41
// (74 VGPRs, 6 waves), 8 waves with 4 sources 9.2.  One column per lane with
// row factors broadcast from LDS took 11.0.  The two-accumulator forms keep
// their 106 VGPRs: spilling them cost a quarter.
constexpr int kSB = 4;

template <int EPI>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(EPI ? 1 : 7, EPI ? 8 : 7))) void k_tile(DevCfg cfg, EvBufs buf, SmearSpec spec, int acc_sel, int nev, int spread,
                                             const int* order, float* out, KlnTab kt) {
  constexpr int TR = kTileRows, NI = TR / 4;
  constexpr int UR = 4, NU = NI / UR;  // row groups per unit, row units
  constexpr bool TWO = EPI != 0;
  __shared__ TileEntry wl[128];
  __shared__ float4 fx_s[kSB][TR / 4];  // K gx: row q + 4 i at q NI + i
  __shared__ float4 fy_s[kSB][16];      // gy: column c + 16 k at 4 c + k
  const int lane = threadIdx.x, q = lane >> 4, c = lane & 15;
  const TileAt at = tile_at(cfg, buf, nev, spread, order);
  if (at.e < 0) return;
  const int e = at.e, r0 = at.R0, c0 = at.c0;
  // tiles outside the event's source rectangle stay zero
  const bool live = at.col_live && at.x0 < r0 + TR && at.x1 > r0;
  if (!live && spec.sparse) {  // nothing to store: zero centre-of-mass partials only
    if (spec.cm_out && lane < 4) spec.cm_out[((size_t)e * at.T + at.tile) * 4 + lane] = 0.0;
    return;
  }
  // exp2 argument -(d_h)^2 kH^2 inv2w2 log2 e with d_h in half-quanta (kH^2 is a power of two)
  const float cq = cfg.inv2w2 * 1.4426950408889634f * (kHf * kHf);
  const float kk = cfg.tile_k;
  const int col = c0 + lane;
  const int ygh = (int)llrint((cfg.ymin + col * cfg.dy) / kH);
  const int rl = lane & (TR - 1), rs = lane / TR;  // row and source of a pass whose factor this lane computes
  const int rowh = (int)llrint((cfg.xmin + (r0 + rl) * cfg.dx) / kH);
  const int4* src = buf.src + (size_t)e * buf.src_cap;
  const int4* swin = buf.swin + (size_t)e * buf.src_cap;

  float acc[NI][4], accA[TWO ? NI : 1][4];  // accA: T_A while the second pass fills acc with T_B
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[i][k] = 0.f;

  for (int pass = 0; pass < (TWO ? 2 : 1); ++pass) {
    if (TWO && pass == 1) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          accA[TWO ? i : 0][k] = acc[i][k];
          acc[i][k] = 0.f;
        }
    }
    const int want = TWO ? pass : acc_sel;
    const int2 kr = source_range(buf, spec, e, want);
    const int K = live ? kr.y : 0;
    int n = 0;  // selected sources waiting in wl
    for (int sub = kr.x; sub < K || n > 0;) {
      // select until 64 wait or the list ends
      while (sub < K && n < 64) {
        const int k = sub + lane;
        sub += 64;
        TileEntry en{0, 0, 0, 0, 0.f, 0u};
        if (k < K) en = tile_entry<4 * UR, NU>(cfg, spec, src[k], swin[k], want, r0, c0);
        const unsigned long long m = __ballot(en.units != 0u);
        if (en.units) wl[n + __popcll(m & ((1ull << lane) - 1ull))] = en;
        n += __popcll(m);
      }
      __builtin_amdgcn_wave_barrier();
      const int take = min(n, 64);
      const TileEntry me = wl[lane];
      for (int g = 0; g < take; g += kSB) {
        const int ng = min(kSB, take - g);
#pragma unroll
        for (int p = 0; p < kSB; p += 64 / TR) {
          if (p >= ng) break;
          const int2 ex = *reinterpret_cast<const int2*>(&wl[g + p + rs].xh);
          const float dx = (float)(rowh - ex.x);
          const int xlo = ex.y & 0xffff, xhi = ex.y >> 16;
          const float gx = kk * __builtin_amdgcn_exp2f(-(dx * dx) * cq);
          reinterpret_cast<float*>(fx_s[p + rs])[(rl & 3) * NI + (rl >> 2)] =
              (r0 + rl >= xlo && r0 + rl < xhi) ? gx : 0.f;
        }
#pragma unroll
        for (int u = 0; u < kSB; ++u) {
          if (u >= ng) break;
          const int yh = __builtin_amdgcn_readlane(me.yh, g + u), yw = __builtin_amdgcn_readlane(me.yw, g + u);
          const int ylo = yw & 0xffff, yhi = yw >> 16;
          const float dy = (float)(ygh - yh);
          reinterpret_cast<float*>(fy_s[u])[4 * c + q] =
              (col >= ylo && col < yhi) ? __builtin_amdgcn_exp2f(-(dy * dy) * cq) : 0.f;
        }
        __builtin_amdgcn_wave_barrier();
        for (int u = 0; u < ng; ++u) {
          const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(me.w), g + u));
          const unsigned um = __builtin_amdgcn_readlane(me.units, g + u);
          float x[NI];
          const float* fx = reinterpret_cast<const float*>(fx_s[u]) + q * NI;
#pragma unroll
          for (int i = 0; i < NI; ++i) x[i] = fx[i];
          const float4 y4 = fy_s[u][c];
          const float y[4] = {y4.x, y4.y, y4.z, y4.w};
#pragma unroll
          for (int b = 0; b < 4 * NU; ++b) {
            if ((um >> b) & 1u) {
#pragma unroll
              for (int i = (b >> 2) * UR; i < ((b >> 2) + 1) * UR; ++i)
                acc[i][b & 3] = fmaf(x[i] * y[b & 3], w, acc[i][b & 3]);
            }
          }
        }
        __builtin_amdgcn_wave_barrier();
      }
      n -= take;
      if (lane < n) wl[lane] = wl[64 + lane];  // n <= 63 are left
      __builtin_amdgcn_wave_barrier();
    }
  }
  // lane = column again: a[4 i + j] is row 4 i + j
  float a[TR], aA[TWO ? TR : 1];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    transpose_groups(acc[i]);
    if constexpr (TWO) transpose_groups(accA[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a[4 * i + j] = acc[i][j];
      if constexpr (TWO) aA[4 * i + j] = accA[i][j];
    }
  }
  tile_finish<TR, EPI>(cfg, buf, at, r0, live, a, aA, kt, out);
  if (spec.cm_out) {
    double s0 = 0.0, s1 = 0.0;
    column_sums<TR>(cfg, at, r0, a, s0, s1);
    tile_cm(cfg, at, s0, s1, spec.cm_out);
  }
}

// ---- four waves of 8 rows per tile, between the two: the workgroup selects
// 256 sources at a time and shares the factors of kGB4 sources, double-
// buffered, one barrier per kGB4 sources.
constexpr int kGB4 = 16;

template <int EPI>
__global__ __launch_bounds__(256) void k_tile4(DevCfg cfg, EvBufs buf, SmearSpec spec, int acc_sel, int nev, int spread,
                                               const int* order, float* out, KlnTab kt) {
  constexpr int NW = 4, TR = kTileRows / NW, NI = TR / 4;
  constexpr bool TWO = EPI != 0;
  __shared__ TileEntry wl[256];
  __shared__ float fx_s[2][kGB4][kTileRows];  // K gx: row 8 v + q + 4 i at 8 v + 2 q + i
  __shared__ float4 fy_s[2][kGB4][16];        // gy: column c + 16 k at 4 c + k
  __shared__ int cnt_s[NW];
  __shared__ double cm_s[2][64];
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), q = lane >> 4, c = lane & 15;
  const TileAt at = tile_at(cfg, buf, nev, spread, order);
  if (at.e < 0) return;
  const int e = at.e, R0 = at.R0, r0 = R0 + TR * wv, c0 = at.c0;
  const bool live = at.col_live && at.x0 < R0 + kTileRows && at.x1 > R0;
  if (!live && spec.sparse) {  // uniform over the workgroup
    if (spec.cm_out && t < 4) spec.cm_out[((size_t)e * at.T + at.tile) * 4 + t] = 0.0;
    return;
  }
  const float cq = cfg.inv2w2 * 1.4426950408889634f * (kHf * kHf);
  const float kk = cfg.tile_k;
  const int col = c0 + lane, row = R0 + (t & 31);  // of the factors this thread computes
  const int ygh = (int)llrint((cfg.ymin + col * cfg.dy) / kH);
  const int rowh = (int)llrint((cfg.xmin + row * cfg.dx) / kH);
  const int fxi = (t & 24) + 2 * (t & 3) + ((t >> 2) & 1);
  const int4* src = buf.src + (size_t)e * buf.src_cap;
  const int4* swin = buf.swin + (size_t)e * buf.src_cap;

  float acc[NI][4], accA[TWO ? NI : 1][4];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[i][k] = 0.f;

  for (int pass = 0; pass < (TWO ? 2 : 1); ++pass) {
    if (TWO && pass == 1) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          accA[TWO ? i : 0][k] = acc[i][k];
          acc[i][k] = 0.f;
        }
    }
    const int want = TWO ? pass : acc_sel;
    const int2 kr = source_range(buf, spec, e, want);
    const int k0 = kr.x, K = live ? kr.y : 0;
    int4 ps = make_int4(0, 0, 0, 0), pw = ps;  // this thread's source of the next 256
    if (k0 + t < K) {
      ps = src[k0 + t];
      pw = swin[k0 + t];
    }
    for (int sub = k0; sub < K; sub += 256) {
      TileEntry en{0, 0, 0, 0, 0.f, 0u};
      if (sub + t < K) en = tile_entry<TR, NW>(cfg, spec, ps, pw, want, R0, c0);
      if (sub + 256 + t < K) {
        ps = src[sub + 256 + t];
        pw = swin[sub + 256 + t];
      }
      const unsigned long long m = __ballot(en.units != 0u);
      __syncthreads();  // the entries and counts of the last round are read
      if (lane == 0) cnt_s[wv] = __popcll(m);
      __syncthreads();
      int n = 0, at_n = 0;
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        if (v == wv) at_n = n;
        n += cnt_s[v];
      }
      if (en.units) wl[at_n + __popcll(m & ((1ull << lane) - 1ull))] = en;
      __syncthreads();
      for (int g = 0; g < n; g += kGB4) {
        const int b = (g / kGB4) & 1, ng = min(kGB4, n - g);
        // factors: rows of 8 sources, then columns of 4 sources, per pass
#pragma unroll
        for (int p = 0; p < kGB4; p += 8) {
          const int s = p + (t >> 5);
          if (s < ng) {
            const int2 ex = *reinterpret_cast<const int2*>(&wl[g + s].xh);
            const float dx = (float)(rowh - ex.x);
            const int xlo = ex.y & 0xffff, xhi = ex.y >> 16;
            const float gx = kk * __builtin_amdgcn_exp2f(-(dx * dx) * cq);
            fx_s[b][s][fxi] = (row >= xlo && row < xhi) ? gx : 0.f;
          }
        }
#pragma unroll
        for (int p = 0; p < kGB4; p += NW) {
          const int s = p + wv;
          if (s < ng) {
            const int2 ey = *reinterpret_cast<const int2*>(&wl[g + s].yh);
            const float dy = (float)(ygh - ey.x);
            const int ylo = ey.y & 0xffff, yhi = ey.y >> 16;
            reinterpret_cast<float*>(fy_s[b][s])[4 * c + q] =
                (col >= ylo && col < yhi) ? __builtin_amdgcn_exp2f(-(dy * dy) * cq) : 0.f;
          }
        }
        // the batch's sources that reach this wave's rows
        const int mine = g + (lane & (kGB4 - 1));
        const float mw = wl[mine].w;
        const unsigned mu = (wl[mine].units >> (4 * wv)) & 15u;
        unsigned mm = (unsigned)__ballot(lane < ng && mu != 0u);
        __syncthreads();
        const auto read = [&](int u, float2& x, float4& y) {
          x = *reinterpret_cast<const float2*>(&fx_s[b][u][TR * wv + 2 * q]);
          y = fy_s[b][u][c];
        };
        float2 xn = make_float2(0.f, 0.f);
        float4 yn = make_float4(0.f, 0.f, 0.f, 0.f);
        int u = mm ? __ffs((int)mm) - 1 : 0;
        if (mm) read(u, xn, yn);
        while (mm) {  // the next source's factors are read while this one is added
          const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mw), u));
          const float2 x = xn;
          const float4 y4 = yn;
          mm &= mm - 1;
          if (mm) {
            u = __ffs((int)mm) - 1;
            read(u, xn, yn);
          }
          const float y[4] = {y4.x, y4.y, y4.z, y4.w};
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            acc[0][k] = fmaf(x.x * y[k], w, acc[0][k]);
            acc[1][k] = fmaf(x.y * y[k], w, acc[1][k]);
          }
        }
      }
    }
  }
  float a[TR], aA[TWO ? TR : 1];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    transpose_groups(acc[i]);
    if constexpr (TWO) transpose_groups(accA[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a[4 * i + j] = acc[i][j];
      if constexpr (TWO) aA[4 * i + j] = accA[i][j];
    }
  }
  tile_finish<TR, EPI>(cfg, buf, at, r0, live, a, aA, kt, out);
  if (!spec.cm_out) return;
  for (int v = 0; v < NW; ++v) {  // each wave goes on from the sums of the rows before its own
    if (wv == v) {
      double s0 = v ? cm_s[0][lane] : 0.0, s1 = v ? cm_s[1][lane] : 0.0;
      column_sums<TR>(cfg, at, r0, a, s0, s1);
      cm_s[0][lane] = s0;
      cm_s[1][lane] = s1;
      if (v == NW - 1) tile_cm(cfg, at, s0, s1, spec.cm_out);
    }
    __syncthreads();
  }
}

// The events of a batch by falling source count (64 classes), so that the
// longest tiles start first and the batch ends without waiting for one of
// them.  The order within a class is free: results do not depend on it.
__global__ __launch_bounds__(1024) void k_tile_order(const int* __restrict__ counts, int nev, int top,
                                                     int* __restrict__ order) {
  __shared__ int cls[64], base[64];
  const int t = threadIdx.x;
  if (t < 64) cls[t] = 0;
  __syncthreads();
  const auto cls_of = [&](int e) { return 63 - min(63, (int)((long long)counts[(size_t)e * 8 + 5] * 64 / (top + 1))); };
  for (int e = t; e < nev; e += 1024) atomicAdd(&cls[cls_of(e)], 1);
  __syncthreads();
  if (t == 0) {
    int s = 0;
    for (int k = 0; k < 64; ++k) {
      base[k] = s;
      s += cls[k];
    }
  }
  __syncthreads();
  for (int e = t; e < nev; e += 1024) order[atomicAdd(&base[cls_of(e)], 1)] = e;
}

// ---- sixteen waves per tile, for batches too small to fill the chip: a
// tile's time is then the chain over its sources, a central event's the
// longest (1,800 sources in one tile).  A wave owns 8 rows x 16 columns, one
// unit of the selection, and adds only the sources that reach it.  The
// workgroup selects 1024 sources at a time (the next 1024 are loaded
// meanwhile) and computes the factors of kGB sources together, double-
// buffered, one barrier per kGB sources.  The sums go through LDS to the four
// waves that store the tile as the one-wave kernel does.
constexpr int kGB = 32;

template <int EPI>
__global__ __launch_bounds__(1024) void k_tile16(DevCfg cfg, EvBufs buf, SmearSpec spec, int acc_sel, int nev,
                                                 int spread, const int* order, float* out, KlnTab kt) {
  constexpr int NW = 16, TR = 8, NT = 64 * NW;
  constexpr bool TWO = EPI != 0;
  __shared__ TileEntry wl[NT];
  __shared__ float fx_s[2][kGB][kTileRows];  // K gx: row 8 v + q + 4 i at 8 v + 2 q + i
  __shared__ float fy_s[2][kGB][64];         // gy
  __shared__ int cnt_s[NW];
  __shared__ float sum_s[TWO ? 2 : 1][kTileRows][64];
  __shared__ double cm_s[2][64];
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), q = lane >> 4, c = lane & 15;
  const int wr = wv >> 2, wc = wv & 3;  // the wave's 8 rows and 16 columns: unit 4 wr + wc = wv
  const TileAt at = tile_at(cfg, buf, nev, spread, order);
  if (at.e < 0) return;
  const int e = at.e, R0 = at.R0, c0 = at.c0;
  const bool live = at.col_live && at.x0 < R0 + kTileRows && at.x1 > R0;
  if (!live && spec.sparse) {  // uniform over the workgroup
    if (spec.cm_out && t < 4) spec.cm_out[((size_t)e * at.T + at.tile) * 4 + t] = 0.0;
    return;
  }
  const float cq = cfg.inv2w2 * 1.4426950408889634f * (kHf * kHf);
  const float kk = cfg.tile_k;
  const int col = c0 + lane, row = R0 + (t & 31);  // of the factors this thread computes
  const int ygh = (int)llrint((cfg.ymin + col * cfg.dy) / kH);
  const int rowh = (int)llrint((cfg.xmin + row * cfg.dx) / kH);
  const int fxi = (t & 24) + 2 * (t & 3) + ((t >> 2) & 1);
  const int4* src = buf.src + (size_t)e * buf.src_cap;
  const int4* swin = buf.swin + (size_t)e * buf.src_cap;

  for (int pass = 0; pass < (TWO ? 2 : 1); ++pass) {
    float acc0 = 0.f, acc1 = 0.f;  // rows q and q + 4 of the wave's 8
    const int want = TWO ? pass : acc_sel;
    const int2 kr = source_range(buf, spec, e, want);
    const int k0 = kr.x, K = live ? kr.y : 0;
    int4 ps = make_int4(0, 0, 0, 0), pw = ps;  // this thread's source of the next 1024
    if (k0 + t < K) {
      ps = src[k0 + t];
      pw = swin[k0 + t];
    }
    for (int sub = k0; sub < K; sub += NT) {
      TileEntry en{0, 0, 0, 0, 0.f, 0u};
      if (sub + t < K) en = tile_entry<TR, 4>(cfg, spec, ps, pw, want, R0, c0);
      if (sub + NT + t < K) {
        ps = src[sub + NT + t];
        pw = swin[sub + NT + t];
      }
      const unsigned long long m = __ballot(en.units != 0u);
      __syncthreads();  // the entries and counts of the last round are read
      if (lane == 0) cnt_s[wv] = __popcll(m);
      __syncthreads();
      int n = 0, at_n = 0;
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        if (v == wv) at_n = n;
        n += cnt_s[v];
      }
      if (en.units) wl[at_n + __popcll(m & ((1ull << lane) - 1ull))] = en;
      __syncthreads();
      for (int g = 0; g < n; g += kGB) {
        const int b = (g / kGB) & 1, ng = min(kGB, n - g);
        // factors: rows of 32 sources in one pass, columns of 16 per pass
        {
          const int s = t >> 5;
          if (s < ng) {
            const int2 ex = *reinterpret_cast<const int2*>(&wl[g + s].xh);
            const float dx = (float)(rowh - ex.x);
            const int xlo = ex.y & 0xffff, xhi = ex.y >> 16;
            const float gx = kk * __builtin_amdgcn_exp2f(-(dx * dx) * cq);
            fx_s[b][s][fxi] = (row >= xlo && row < xhi) ? gx : 0.f;
          }
        }
#pragma unroll
        for (int p = 0; p < kGB; p += NW) {
          const int s = p + wv;
          if (s < ng) {
            const int2 ey = *reinterpret_cast<const int2*>(&wl[g + s].yh);
            const float dy = (float)(ygh - ey.x);
            const int ylo = ey.y & 0xffff, yhi = ey.y >> 16;
            fy_s[b][s][lane] = (col >= ylo && col < yhi) ? __builtin_amdgcn_exp2f(-(dy * dy) * cq) : 0.f;
          }
        }
        // the batch's sources that reach this wave's unit
        const int mine = g + (lane & (kGB - 1));
        const float mw = wl[mine].w;
        unsigned mm = (unsigned)__ballot(lane < ng && ((wl[mine].units >> wv) & 1u));
        __syncthreads();
        while (mm) {  // four sources' factors are read before they are added, in order
          float2 x[4];
          float y[4], w[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            if (mm) {
              const int u = __ffs((int)mm) - 1;
              mm &= mm - 1;
              x[v] = *reinterpret_cast<const float2*>(&fx_s[b][u][TR * wr + 2 * q]);
              y[v] = fy_s[b][u][16 * wc + c];
              w[v] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mw), u));
            } else {
              x[v] = make_float2(0.f, 0.f);
              y[v] = w[v] = 0.f;
            }
          }
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            acc0 = fmaf(x[v].x * y[v], w[v], acc0);
            acc1 = fmaf(x[v].y * y[v], w[v], acc1);
          }
        }
      }
    }
    sum_s[TWO ? pass : 0][TR * wr + q][16 * wc + c] = acc0;
    sum_s[TWO ? pass : 0][TR * wr + q + 4][16 * wc + c] = acc1;
  }
  __syncthreads();
  const int r0 = R0 + TR * wv;
  float a[TR] = {};
  if (wv < 4) {  // wave v stores rows 8 v .. 8 v + 7
    float aA[TWO ? TR : 1];
#pragma unroll
    for (int r = 0; r < TR; ++r) {
      a[r] = sum_s[TWO ? 1 : 0][TR * wv + r][lane];
      if constexpr (TWO) aA[r] = sum_s[0][TR * wv + r][lane];
    }
    tile_finish<TR, EPI>(cfg, buf, at, r0, live, a, aA, kt, out);
  }
  if (!spec.cm_out) return;
  for (int v = 0; v < 4; ++v) {  // as in k_tile4
    if (wv == v) {
      double s0 = v ? cm_s[0][lane] : 0.0, s1 = v ? cm_s[1][lane] : 0.0;
      column_sums<TR>(cfg, at, r0, a, s0, s1);
      cm_s[0][lane] = s0;
      cm_s[1][lane] = s1;
      if (v == 3) tile_cm(cfg, at, s0, s1, spec.cm_out);
    }
    __syncthreads();
  }
}

int tile_units(const DevCfg& cfg) { return ((cfg.nx + kTileRows - 1) / kTileRows) * ((cfg.ny + 63) / 64); }

// About how many sources a central event's list holds: the nucleons that n
// collisions wound and, where the spec has the pairs, the n pairs; n = 1.5 A B
// sigma / (pi R^2) of the larger radius (a sphere is 1.5 times as thick at its
// centre as on average).  Pb+Pb 3,400 with pairs and 416 without, 63+63 810
// and 126, 20+20 170 and 40, d+Au 60 and 30, p+Pb 30 and 15.  The nuclei are
// the context's, the largest of a mixed batch.
static double central_list(const DevCfg& cfg, const SmearSpec& s) {
  const NucSys &p = cfg.nuc[0], &t = cfg.nuc[1];
  const double R = std::max(1.0, (double)std::max(p.R, t.R));
  const double n = std::min((double)p.A * t.A, 1.5 * p.A * t.A * (double)cfg.hit_n * (kQ * kQ) / (R * R));
  return std::min((double)p.A, n) + std::min((double)t.A, n) + (s.enabled[kSrcPair] ? n : 0.0);
}

// Waves per tile.  Variants 1, 2, 3 (smc_set_tile_variant) are one, four and
// sixteen; 0 chooses by the number of tiles and the length of a central list.
// us with 1 / 4 / 16 waves per batch of events of 261^2 cells (45 tiles):
//   Pb+Pb, pairs    30 events 404 / 196 / 105, 100 453 / 221 / 129, 200 468 / 225 / 233,
//                   1000 514 / 342 / 1091, 2000 543 / 652 / 2168
//   Pb+Pb, MC-KLN   30 events 89 / 47 / 40, 100 97 / 52 / 96, 500 105 / 109 / 401,
//                   1000 163 / 191 / 768
//   20+20, pairs    30 events 38 / 26 / 23, 200 44 / 28 / 72, 500 48 / 44 / 158,
//                   1000 50 / 71 / 300
//   p+Pb, pairs     8 events 17 / 12 / 11, 200 24 / 22 / 59, 500 30 / 36 / 133,
//                   1000 39 / 58 / 255
//   p+Pb, MC-KLN    8 events 26 / 15 / 15, 200 37 / 29 / 82, 500 47 / 49 / 188,
//                   1000 70 / 81 / 359
// A short list leaves sixteen waves nothing but their barriers.
constexpr double kShortList = 100.0, kLongList = 700.0;

static int waves_of(const DevCfg& cfg, const SmearSpec& s, int nev) {
  constexpr int kWaves[kTileVariants] = {0, 1, 4, 16};
  const long long tiles = (long long)tile_units(cfg) * nev;
  if (cfg.tile_variant > 0 && cfg.tile_variant < kTileVariants) {
    // a launch has fewer than 2^32 work-items: batches beyond that for the
    // variant's shape (93,000 events of 45 tiles with sixteen waves) take the
    // next smaller one; one wave per tile fits any batch that memory holds
    int waves = kWaves[cfg.tile_variant];
    while (waves > 1 && (tiles + 8 * tile_units(cfg)) * 64 * waves >= (1LL << 32)) waves /= 4;
    return waves;
  }
  const double list = central_list(cfg, s);
  if (list < kShortList) return tiles <= 9000 ? 4 : 1;
  const bool heavy = list >= kLongList;
  return tiles <= (heavy ? 9000 : 2200) ? 16 : (tiles <= (heavy ? 58000 : 20000) ? 4 : 1);
}

// Longest events first: 1000 Pb+Pb events 735 -> 504 us with one wave per tile,
// 543 -> 362 with four; 16,000 events 3.2 -> 2.9 ms.  One workgroup orders
// 32,768 events in about 60 us; larger batches lose less to their last tiles.
// Events of short lists are too alike to gain it back (p+Pb: 5 of 25 us at 200
// events, 60 of 470 at 20,000).
static bool ordered(const DevCfg& cfg, const SmearSpec& s, int nev) {
  return nev >= 16 && nev <= 32768 && central_list(cfg, s) >= kShortList;
}

template <int EPI>
static void launch_shape(const DevCfg& cfg, const EvBufs& b, const SmearSpec& s, int acc_sel, int nev, float* out,
                         const KlnTab& kt, hipStream_t st) {
  const int waves = waves_of(cfg, s, nev);
  const int spread = nev < 64;  // 8 events per XCD keep its 32 CUs busy
  const int* order = ordered(cfg, s, nev) ? b.order : nullptr;
  // one dimension: tiles x events; with an event's tiles on one XCD, events
  // padded to a multiple of the 8 XCDs
  const dim3 grid((unsigned)tile_units(cfg) * (spread ? (unsigned)nev : (unsigned)((nev + 7) / 8 * 8)));
  if (waves == 16)
    hipLaunchKernelGGL(k_tile16<EPI>, grid, dim3(1024), 0, st, cfg, b, s, acc_sel, nev, spread, order, out, kt);
  else if (waves == 4)
    hipLaunchKernelGGL(k_tile4<EPI>, grid, dim3(256), 0, st, cfg, b, s, acc_sel, nev, spread, order, out, kt);
  else
    hipLaunchKernelGGL(k_tile<EPI>, grid, dim3(64), 0, st, cfg, b, s, acc_sel, nev, spread, order, out, kt);
}

static void launch_order(const DevCfg& cfg, const EvBufs& b, const SmearSpec& s, int nev, hipStream_t st) {
  if (ordered(cfg, s, nev))
    hipLaunchKernelGGL(k_tile_order, dim3(1), dim3(1024), 0, st, b.counts, nev, 2048, b.order);
}

// The fused MC-KLN launch (its centre-of-mass partials have tile_units(cfg)
// units).
int launch_tile_kln(const DevCfg& cfg, const EvBufs& b, const SmearSpec& s, int nev, float* out,
                    const double* table, int tmax, double dT, void* stream) {
  if (nev <= 0) return 0;
  if (!(cfg.tile_k > 0.f && cfg.tile_w > 0.f && cfg.tile_out > 0.f) || !table || tmax < 3 || !(dT > 0))
    return (int)hipErrorInvalidValue;
  launch_order(cfg, b, s, nev, (hipStream_t)stream);
  launch_shape<1>(cfg, b, s, 0, nev, out, KlnTab{table, tmax, dT}, (hipStream_t)stream);
  return (int)hipGetLastError();
}

// Cells outside each event's source rectangle set to zero (the grid of a
// sparse launch, completed before whole grids are read).
__global__ __launch_bounds__(256) void k_zero_outside(float* grid, const int* counts, int nx, int ny) {
  const int e = blockIdx.y;
  const int rx = counts[(size_t)e * 8 + 6], ry = counts[(size_t)e * 8 + 7];
  const int x0 = rx & 0xffff, x1 = rx >> 16, y0 = ry & 0xffff, y1 = ry >> 16;
  float* g = grid + (size_t)e * nx * ny;
  const int n = nx * ny;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const int ix = i / ny, iy = i - ix * ny;
    if (ix < x0 || ix >= x1 || iy < y0 || iy >= y1) g[i] = 0.f;
  }
}

int launch_zero_outside(float* g, const int* counts, int nx, int ny, int nev, void* stream) {
  if (nev <= 0) return 0;
  const int per = (nx * ny + 255) / 256;
  const dim3 grid((unsigned)(per < 64 ? per : 64), (unsigned)nev);
  hipLaunchKernelGGL(k_zero_outside, grid, dim3(256), 0, (hipStream_t)stream, g, counts, nx, ny);
  return (int)hipGetLastError();
}

int launch_tile(const DevCfg& cfg, const EvBufs& b, const SmearSpec& s, int nev, float* out0, float* out1,
                void* stream) {
  if (nev <= 0) return 0;
  if (!(cfg.tile_k > 0.f && cfg.tile_w > 0.f && cfg.tile_out > 0.f)) return (int)hipErrorInvalidValue;
  hipStream_t st = (hipStream_t)stream;
  const KlnTab none{nullptr, 0, 1.0};
  launch_order(cfg, b, s, nev, st);
  if (s.combine == 1) {  // sqrt(T_A T_B) in one launch, with the partials of the combined grid
    launch_shape<2>(cfg, b, s, 0, nev, out0, none, st);
    return (int)hipGetLastError();
  }
  SmearSpec s1 = s;  // partials only for a single accumulator
  if (s.combine != 0) s1.cm_out = nullptr;
  launch_shape<0>(cfg, b, s1, 0, nev, out0, none, st);
  if (s.combine != 0) launch_shape<0>(cfg, b, s1, 1, nev, out1, none, st);
  return (int)hipGetLastError();
}

}  // namespace smc
