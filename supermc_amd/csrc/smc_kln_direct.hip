// smc_kln_direct.hip -- MC-KLN dN/dy by the k_T-factorised quadrature in
// every cell, FP32 (KLNModel.cpp:97-125, :219-277, :360-399; the factorised
// integrand and node tables of smc_kln.hip):
//   sum_pT P / (alpha(a) alpha(b)) sum_n c_n min(1, a u_n) min(1, b v_n)
// with a = T_A g(pT), b = T_B g(pT).  The cells with T_A, T_B > 0 are
// compacted first, then one lane per such cell; the node data are read
// through the scalar unit (uniform addresses); FP64 only for the per-pT
// sum.  Each node is taken as c_n min(1/a, u_n) min(1/b, v_n), the
// sum times a b once per pT node: two minima, a multiply and an FMA.  The
// file is built without NaN semantics (-fno-honor-nans), so that a minimum
// of a value read through the scalar unit is one instruction (with them
// the compiler first quiets it as a possible signalling NaN); the inputs
// are the finite T_A, T_B grids and the host's finite node tables.
//
// The node sum F(x, y) = sum_n c_n min(x, u_n) min(y, v_n) at x = 1/a,
// y = 1/b is bilinear between consecutive u_n and v_n: its values at those
// breakpoints (one table per pT node, built once from the node tables) give
// every F by one bilinear interpolation, with no approximation beyond
// rounding.  A cell then costs two searches and one 16-byte table read per
// pT node instead of a pass over the nodes (k_kln_interp); node tables too
// large for that are summed node by node (k_kln_direct).
#include <algorithm>

#include "smc_device.h"

namespace smc {

__device__ __forceinline__ float alpha_s_f(float q2, float lq2, float amax, float inv_beta0) {
  if (q2 <= lq2) return amax;
  return fminf(amax, inv_beta0 / logf(q2 / lq2));
}

// dN/dy of cell i from its T_A = A, T_B = B (both > 0).
// node layout: ptf[i] = {P, g}, nodes[i * nn + n] = {c, u, v}, nn a multiple of 16
__device__ __forceinline__ float kln_direct_cell(float A, float B, const float2* ptf, const float4* nodes, int npt,
                                                 int nn, const KlnConst& kc) {
  const float lq2 = (float)kc.lq2, amax = (float)kc.amax, ib0 = (float)kc.inv_beta0;
  double sum = 0.0;
  for (int p = 0; p < npt; ++p) {
    const float2 pg = ptf[p];  // {P, g}
    const float a = A * pg.y, b = B * pg.y;
    const float ia = 1.f / a, ib = 1.f / b;
    // sixteen nodes per step (the table is padded to a multiple of 16 with
    // zero nodes) into four sums; the node offsets are wave-uniform, so a
    // step's loads go out together through the scalar unit
    const int n0 = __builtin_amdgcn_readfirstlane(p * nn);
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int n = n0; n < n0 + nn; n = __builtin_amdgcn_readfirstlane(n + 16)) {
      const float4* q = nodes + n;
      float4 v[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) v[k] = q[k];
#pragma unroll
      for (int k = 0; k < 16; ++k) s[k & 3] = fmaf(v[k].x, fminf(ia, v[k].y) * fminf(ib, v[k].z), s[k & 3]);
    }
    const float inv = 1.f / (alpha_s_f(a, lq2, amax, ib0) * alpha_s_f(b, lq2, amax, ib0));
    sum += (double)pg.x * (double)(((s[0] + s[1]) + (s[2] + s[3])) * (a * b) * inv);
  }
  return (float)sum;
}

// The cells with T_A, T_B > 0 of the batch, compacted (in no fixed order:
// each cell is computed on its own) into list[0 .. *count); the others get
// dN/dy = 0 here.  *count starts at 0 (k_kln_count_reset).  A workgroup
// takes KLN_ACT_CELLS consecutive cells (KLN_ACT_PER per lane, coalesced)
// and reserves its share of the list with one atomic.
constexpr int KLN_ACT_PER = 8;
constexpr int KLN_ACT_CELLS = 256 * KLN_ACT_PER;
__global__ __launch_bounds__(256) void k_kln_active(const float* __restrict__ ta, const float* __restrict__ tb,
                                                    float* __restrict__ out, size_t ncell, unsigned* __restrict__ list,
                                                    unsigned* count) {
  __shared__ unsigned woff[4][KLN_ACT_PER];  // per wave and step: its count, then its offset in the block's share
  __shared__ unsigned base_s;
  const size_t b0 = (size_t)blockIdx.x * KLN_ACT_CELLS;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  unsigned long long m[KLN_ACT_PER];
#pragma unroll
  for (int k = 0; k < KLN_ACT_PER; ++k) {
    const size_t i = b0 + (size_t)k * 256 + threadIdx.x;
    bool act = false;
    if (i < ncell) {
      act = ta[i] > 0.f && tb[i] > 0.f;
      if (!act) out[i] = 0.f;
    }
    m[k] = __ballot(act);
  }
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < KLN_ACT_PER; ++k) woff[w][k] = (unsigned)__popcll(m[k]);
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned tot = 0;
    for (int ww = 0; ww < 4; ++ww)
      for (int k = 0; k < KLN_ACT_PER; ++k) {
        const unsigned c = woff[ww][k];
        woff[ww][k] = tot;
        tot += c;
      }
    base_s = tot ? atomicAdd(count, tot) : 0u;
  }
  __syncthreads();
  const unsigned base = base_s;
  const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
  for (int k = 0; k < KLN_ACT_PER; ++k)
    if ((m[k] >> lane) & 1ull)
      list[base + woff[w][k] + (unsigned)__popcll(m[k] & below)] = (unsigned)(b0 + (size_t)k * 256 + threadIdx.x);
}

__global__ void k_kln_count_reset(unsigned* count) { *count = 0u; }

// dN/dy of the listed cells: each wave takes 64 consecutive list entries
// per step (full waves of active cells whatever the shape of the active
// region).  The loop is uniform over the wave -- the last step's spare
// lanes recompute the last entry and store nothing -- and the pointers
// are __restrict__ (the node tables cannot alias the stores), so the node
// loop keeps its scalar loads.
__global__ __launch_bounds__(256) void k_kln_direct(const float* __restrict__ ta, const float* __restrict__ tb,
                                                    float* __restrict__ out, const unsigned* __restrict__ list,
                                                    const unsigned* __restrict__ count,
                                                    const float2* __restrict__ ptf, const float4* __restrict__ nodes,
                                                    int npt, int nn, KlnConst kc) {
  const unsigned n = __builtin_amdgcn_readfirstlane(*count);
  const unsigned lane = threadIdx.x & 63;
  const unsigned wave = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const unsigned nwaves = (gridDim.x * blockDim.x) >> 6;
  for (unsigned j0 = 64 * wave; j0 < n; j0 += 64 * nwaves) {
    const unsigned j = j0 + lane;
    const unsigned i = list[j < n ? j : n - 1];
    const float v = kln_direct_cell(ta[i], tb[i], ptf, nodes, npt, nn, kc);
    if (j < n) out[i] = v;
  }
}

// ---- breakpoint tables
// Per pT node p: bu[p][nn + 1] = {0, u sorted}, bv[p][nn + 1] = {0, v sorted}
// and the nodes in u order with doubles {c, u, v}.  One workgroup per
// (p, axis); a node's rank is its count of smaller values (ties by index).
__global__ __launch_bounds__(256) void k_kln_rank(const double4* __restrict__ nodes, int nn, float* __restrict__ bu,
                                                  float* __restrict__ bv, double4* __restrict__ sorted) {
  __shared__ float val[256];
  const int p = blockIdx.x, axis = blockIdx.y, t = threadIdx.x;
  const double4* q = nodes + (size_t)p * nn;
  float* bp = (axis ? bv : bu) + (size_t)p * (nn + 1);
  if (t == 0) bp[0] = 0.f;
  for (int k0 = 0; k0 < nn; k0 += 256) {  // uniform bounds: every thread meets the barriers
    const int k = k0 + t;
    const double4 nd = k < nn ? q[k] : make_double4(0, 0, 0, 0);
    const float x = (float)(axis ? nd.z : nd.y);
    int rank = 0;
    for (int m0 = 0; m0 < nn; m0 += 256) {
      __syncthreads();
      if (m0 + t < nn) val[t] = (float)(axis ? q[m0 + t].z : q[m0 + t].y);
      __syncthreads();
      const int n = min(256, nn - m0);
      for (int m = 0; m < n; ++m) rank += val[m] < x || (val[m] == x && m0 + m < k);
    }
    if (k < nn) {
      bp[1 + rank] = x;
      if (axis == 0) sorted[(size_t)p * nn + rank] = make_double4(nd.x, (double)x, (double)(float)nd.z, 0.0);
    }
  }
}

// tab[p][i][j] = {F(bu_i, bv_j), F(bu_i+1, bv_j)}, i <= nn, j <= nn + 1 (row
// nn + 1 and column nn + 1 repeat the last: F is constant beyond the last
// breakpoint).  One lane per column walks up the rows in FP64 with
// F(bu_i, y) = sum_{k <= i} c u min(y, v) + bu_i sum_{k > i} c min(y, v).
__global__ __launch_bounds__(64) void k_kln_breaks(const double4* __restrict__ sorted, const float* __restrict__ bv,
                                                   int nn, float2* __restrict__ tab) {
  __shared__ double4 nd[64];
  const int p = blockIdx.y, j = blockIdx.x * 64 + threadIdx.x, cols = nn + 2;
  const double4* q = sorted + (size_t)p * nn;
  const double y = (double)bv[(size_t)p * (nn + 1) + min(j, nn)];
  float2* o = tab + (size_t)p * (nn + 1) * cols + j;
  double below = 0.0, above = 0.0;
  float prev = 0.f;  // F(0, y) = 0
  for (int pass = 0; pass < 2; ++pass) {
    for (int k0 = 0; k0 < nn; k0 += 64) {
      __syncthreads();
      if (k0 + (int)threadIdx.x < nn) nd[threadIdx.x] = q[k0 + threadIdx.x];
      __syncthreads();
      const int n = min(64, nn - k0);
      for (int k = 0; k < n; ++k) {
        const double4 v = nd[k];
        const double cm = v.x * fmin(y, v.z);
        if (pass == 0) {
          above += cm;
          continue;
        }
        above -= cm;
        below = fma(cm, v.y, below);
        const float f = (float)fma(v.y, above, below);
        if (j < cols) o[(size_t)(k0 + k) * cols] = make_float2(prev, f);
        prev = f;
      }
    }
  }
  if (j < cols) o[(size_t)nn * cols] = make_float2(prev, prev);
}

// dN/dy of the listed cells from the breakpoint tables.  Four waves share
// 64 R cells; wave g takes the g-th quarter of the pT nodes, so that a small
// batch still fills the chip, and the four partial sums are added in wave
// order whatever the batch.  A wave keeps the breakpoints of its pT node in
// LDS (the searches are 10 dependent reads each at 768 nodes; from LDS they
// cost a tenth of what they would through the texture path) and reads one
// float4 (both rows, two columns) per cell.  R cells per lane: the 2 R
// searches run in step, so their LDS reads overlap (one search after the
// other took 659 us at the size below, together 430 us).
// Bound by VALU issue (0.243 instructions per SIMD and cycle, as many as a chain
// of FMAs; a CU issues an LDS instruction every nine cycles).  150 Pb+Pb events of
// 261^2 cells, 32 x 32 x 48 nodes: 430 us; summed node by node 3975 us
// (four VALU per node term, 24,576 terms per cell).
constexpr int KLN_R = 4;
__global__ __launch_bounds__(256) void k_kln_interp(const float* __restrict__ ta, const float* __restrict__ tb,
                                                    float* __restrict__ out, const unsigned* __restrict__ list,
                                                    const unsigned* __restrict__ count,
                                                    const float2* __restrict__ ptf, const float* __restrict__ bu,
                                                    const float* __restrict__ bv, const float2* __restrict__ tab,
                                                    int npt, int nn, KlnConst kc) {
  extern __shared__ float bp[];  // [4 waves][2][nn + 1], then the partial sums
  const unsigned n = __builtin_amdgcn_readfirstlane(*count);
  const int lane = threadIdx.x & 63, g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float* xu = bp + g * 2 * (nn + 1);
  float* xv = xu + nn + 1;
  double* part = reinterpret_cast<double*>(bp + 8 * (nn + 1));  // [4][KLN_R * 64], 8-byte aligned
  const float lq2 = (float)kc.lq2, amax = (float)kc.amax, ib0 = (float)kc.inv_beta0;
  const int p0 = npt * g / 4, p1 = npt * (g + 1) / 4;
  const int cols = nn + 2;
  for (unsigned j0 = blockIdx.x * (64u * KLN_R); j0 < n; j0 += gridDim.x * (64u * KLN_R)) {
    float A[KLN_R], B[KLN_R];
    double sum[KLN_R];
    unsigned cell[KLN_R];
#pragma unroll
    for (int r = 0; r < KLN_R; ++r) {
      const unsigned j = j0 + 64u * r + lane;
      cell[r] = list[j < n ? j : n - 1];
      A[r] = ta[cell[r]];
      B[r] = tb[cell[r]];
      sum[r] = 0.0;
    }
    for (int p = p0; p < p1; ++p) {
      const float2 pg = ptf[p];  // {P, g}
      __builtin_amdgcn_wave_barrier();
      for (int k = lane; k <= nn; k += 64) {
        xu[k] = bu[(size_t)p * (nn + 1) + k];
        xv[k] = bv[(size_t)p * (nn + 1) + k];
      }
      __builtin_amdgcn_wave_barrier();
      const float2* tp = tab + (size_t)p * (nn + 1) * cols;
      // the last i with xu[i] <= 1/a (xu[0] = 0) and j alike, all searches of
      // the wave's cells in step: their LDS reads overlap
      float ia[KLN_R], ib[KLN_R];
      int iu[KLN_R], iv[KLN_R];
#pragma unroll
      for (int r = 0; r < KLN_R; ++r) {
        ia[r] = 1.f / (A[r] * pg.y);
        ib[r] = 1.f / (B[r] * pg.y);
        iu[r] = iv[r] = 0;
      }
      for (int len = nn + 1; len > 1;) {
        const int half = len >> 1;
        len -= half;
#pragma unroll
        for (int r = 0; r < KLN_R; ++r) {
          iu[r] = xu[iu[r] + half] <= ia[r] ? iu[r] + half : iu[r];
          iv[r] = xv[iv[r] + half] <= ib[r] ? iv[r] + half : iv[r];
        }
      }
#pragma unroll
      for (int r = 0; r < KLN_R; ++r) {
        const float a = A[r] * pg.y, b = B[r] * pg.y;
        const int i = iu[r], j = iv[r];
        const float u0 = xu[i], u1 = xu[min(i + 1, nn)], v0 = xv[j], v1 = xv[min(j + 1, nn)];
        const float s = i < nn ? (ia[r] - u0) / (u1 - u0) : 0.f, t = j < nn ? (ib[r] - v0) / (v1 - v0) : 0.f;
        const float2* f = tp + (size_t)i * cols + j;
        const float2 f0 = f[0], f1 = f[1];
        const float lo = fmaf(s, f0.y - f0.x, f0.x), hi = fmaf(s, f1.y - f1.x, f1.x);
        const float F = fmaf(t, hi - lo, lo);
        const float inv = 1.f / (alpha_s_f(a, lq2, amax, ib0) * alpha_s_f(b, lq2, amax, ib0));
        sum[r] += (double)pg.x * (double)(F * (a * b) * inv);
      }
    }
#pragma unroll
    for (int r = 0; r < KLN_R; ++r) part[g * (64 * KLN_R) + 64 * r + lane] = sum[r];
    __syncthreads();
    // the cells' sums: wave g adds the four parts of its quarter
    for (int c = threadIdx.x; c < 64 * KLN_R; c += 256) {
      const unsigned j = j0 + c;
      if (j < n)
        out[list[j]] = (float)(((part[c] + part[64 * KLN_R + c]) + part[128 * KLN_R + c]) + part[192 * KLN_R + c]);
    }
    __syncthreads();
  }
}

size_t kln_breaks_doubles(int npt, int nn) { return (size_t)npt * (nn + 1) * (nn + 2); }

// The interpolation kernel's limits: its breakpoints and partial sums in
// 64 KB of LDS, the tables within 512 MiB (32 x 768 nodes take 151 MB and
// 270 us to build).  Within them interpolating is the faster for any batch:
// even the first one, build included, took 2.4 ms against 5.6 ms for 150
// events with 32 x 768 nodes.
bool kln_breaks_fit(int npt, int nn) {
  return nn >= 1 && nn <= 1536 && kln_breaks_doubles(npt, nn) * sizeof(float2) <= ((size_t)512 << 20);
}

int launch_kln_breaks(const void* nodes_d, int npt, int nn, const KlnBreaks& kb, void* stream) {
  if (!kln_breaks_fit(npt, nn)) return (int)hipErrorInvalidValue;
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_kln_rank, dim3(npt, 2), dim3(256), 0, st, (const double4*)nodes_d, nn, kb.bu, kb.bv, (double4*)kb.sorted);
  hipLaunchKernelGGL(k_kln_breaks, dim3((nn + 2 + 63) / 64, npt), dim3(64), 0, st, (const double4*)kb.sorted, kb.bv, nn,
                     (float2*)kb.tab);
  return (int)hipGetLastError();
}

int launch_kln_direct(const float* ta, const float* tb, float* out, size_t ncell, const void* ptf,
                      const void* nodes, int npt, int nn, const KlnConst& kc, const KlnBreaks& kb, unsigned* list,
                      unsigned* count, void* stream) {
  if (ncell == 0) return 0;
  if (ncell > 0xffffffffull) return (int)hipErrorInvalidValue;  // 32-bit cell indices
  if (nn <= 0 || nn % 16 != 0) return (int)hipErrorInvalidValue;  // the node loop's 16-node steps
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(k_kln_count_reset, dim3(1), dim3(1), 0, st, count);
  hipLaunchKernelGGL(k_kln_active, dim3((unsigned)((ncell + KLN_ACT_CELLS - 1) / KLN_ACT_CELLS)), dim3(256), 0, st,
                     ta, tb, out, ncell, list, count);
  if (kb.tab) {
    if (!kln_breaks_fit(npt, nn)) return (int)hipErrorInvalidValue;
    const size_t shm = (size_t)8 * (nn + 1) * sizeof(float) + (size_t)4 * 64 * KLN_R * sizeof(double);
    const unsigned nb = (unsigned)std::min<size_t>((ncell + 64 * KLN_R - 1) / (64 * KLN_R), 16384);
    hipLaunchKernelGGL(k_kln_interp, dim3(nb), dim3(256), shm, st, ta, tb, out, list, count, (const float2*)ptf,
                       kb.bu, kb.bv, (const float2*)kb.tab, npt, nn, kc);
    return (int)hipGetLastError();
  }
  // 32 workgroups of 256 lanes per CU (several times the waves a CU holds
  // at once), or fewer for a small batch
  const unsigned blocks = (unsigned)std::min<size_t>((ncell + 255) / 256, 8192);
  hipLaunchKernelGGL(k_kln_direct, dim3(blocks), dim3(256), 0, st, ta, tb, out, list, count, (const float2*)ptf,
                     (const float4*)nodes, npt, nn, kc);
  return (int)hipGetLastError();
}

}  // namespace smc
