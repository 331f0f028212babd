// smc_grid64.hip -- the entropy-density grid in FP64 with the reference's
// double arithmetic: MCnucl::setDensity for which_mc_model 5
// (MCnucl.cpp:689-760: (1-alpha)/2 sum_part f T_n + alpha sum_coll f G) and
// 7 (MCnucl.cpp:762-811: sqrt(rho_A rho_B)), participants through
// Particle::getSmoothDensity (Particle.cpp:122-132, 168-174) over their
// boxes, collisions over the +-5w windows with the dc <= 25 w^2 cut.
//
// Per (source, cell) in FP64:
//   participant  f / (2 pi w^2) exp(-d^2 / 2w^2) where sqrt(d^2) <= 5w,
//   collision    f / (2 pi w^2) exp(-d^2 / 2w^2) (alpha + (1 - alpha) aw) where
//                d^2 <= 25 w^2, with aw = 0, or for sub_model 2
//                (MCnucl.cpp:713-717: no participant term) the pair's weight
//                of MCnucl.cpp:345-348,
// d^2 = dx^2 + dy^2 rounded as the reference's x86-64 doubles round it (the file
// is built with -ffp-contract=off), so both cuts take the reference's cells:
// sqrt(d^2) <= 5w is the compare d^2 <= part_max with the largest double whose
// root passes (host).  The exponential factorises, exp(-dx^2/2w^2)
// exp(-dy^2/2w^2): a cell costs an add, a compare and an FMA under its mask
// instead of a square root, a division and an exponential.  The weights f norm
// (1 - alpha)/2 and f norm alpha are folded into the column factors, with what
// their own rounding left: a term is off by its exponentials and one product.
// Terms are added in source order (participants of A and B in wound order,
// pairs in pair order), participants and pairs in sums of their own that meet
// at the end, as in the reference: pairs added on top of the participants' sum
// rounded it 2,000 times more and doubled the error.  Against 80-bit sums of
// the same sources (central events, w 0.35 to 1 fm, relative to the largest
// cell) the error is that of an exponential per term or smaller:
// w = 0.5 fm rms 2.7e-17 and at most 1.0e-15 (2.8e-17 and 1.0e-15 with an
// exponential per term, 5.1e-17 and 1.9e-15 in one sum).
//
// One workgroup of 4 waves per (32 x 64 tile, event), a wave 8 rows, laid out as
// k_tile4 of smc_tile.hip: lane (q, c) holds rows q, q + 4 and columns c + 16 k;
// the workgroup selects 256 sources at a time and shares the factors of 8.
// 250 Au+Au events of 261^2 cells 497 us (2226 us with an exponential per term):
// VALU instructions issue at 57 % of the rate of a chain of FMAs with 2.5 waves
// on a SIMD, the rest is the waits between the factors' exponentials, LDS and
// barriers.
// Tiles outside the event's source rectangle are written as zeros without a
// source pass.
#include "smc_device.h"

namespace smc {

namespace {
constexpr int kGX = 32, kGY = 64, kG64 = 8;

struct Entry64 {
  int xh, xw, yh, yw;
  double w, w_lo;  // weight and what its rounding left
  int chunks;  // the 8-row chunks of the tile that the window meets
};
}  // namespace

template <bool ROOT>
__global__ __launch_bounds__(256) void k_grid64(DevCfg cfg, EvBufs buf, Grid64Const gc, int ev0, double* out) {
  constexpr int NW = 4, TR = kGX / NW;
  __shared__ Entry64 wl[256];
  __shared__ double2 fx_s[2][kG64][kGX];  // {gx, dx^2}: row 8 v + q + 4 i at 8 v + 2 q + i
  __shared__ double2 fy_s[2][kG64][kGY];  // {w gy, dy^2}
  __shared__ int cnt_s[NW];
  const int el = blockIdx.y, e = ev0 + el;
  const int ntx = (cfg.nx + kGX - 1) / kGX;
  const int R0 = (blockIdx.x % ntx) * kGX, c0 = (blockIdx.x / ntx) * kGY;
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), q = lane >> 4, c = lane & 15;
  const int rxp = buf.counts[(size_t)e * 8 + 6], ryp = buf.counts[(size_t)e * 8 + 7];
  const bool live = R0 < (rxp >> 16) && R0 + kGX > (rxp & 0xffff) && c0 < (ryp >> 16) && c0 + kGY > (ryp & 0xffff);
  const int npa = buf.counts[(size_t)e * 8], npart = npa + buf.counts[(size_t)e * 8 + 1];
  const int K = live ? buf.counts[(size_t)e * 8 + 5] : 0;  // uniform over the workgroup
  const int4* src = buf.src + (size_t)e * buf.src_cap;
  const int4* swin = buf.swin + (size_t)e * buf.src_cap;
  const size_t pbase = (size_t)e * cfg.max_pairs;
  const int row = R0 + (t & 31), col = c0 + lane;  // of the factors this thread computes
  const double xg = cfg.xmin + (double)row * cfg.dx, yg = cfg.ymin + (double)col * cfg.dy;
  const int fxi = (t & 24) + 2 * (t & 3) + ((t >> 2) & 1);

  double acc[2][4], acc0[2][4];  // of the pass, of the first pass
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[i][k] = 0.0;
  for (int pass = 0; pass < 2; ++pass) {
    if (pass == 1) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          acc0[i][k] = acc[i][k];
          acc[i][k] = 0.0;
        }
    }
    // model 7 (ROOT): the projectile's participants, then the target's; model
    // 5: the participants (none for sub_model 2), then the pairs (none at
    // alpha = 0)
    const bool pairs = !ROOT && pass == 1;
    const int k0 = pass ? min(ROOT ? npa : npart, K) : 0;
    const int k1 = ROOT ? min(pass ? npart : npa, K) : (pass ? (gc.use_binary ? K : 0) : (gc.uli ? 0 : min(npart, K)));
    const double cut = pairs ? gc.dc_max : gc.part_max;
    for (int sub = k0; sub < k1; sub += 256) {
      const int k = sub + t;
      Entry64 en{0, 0, 0, 0, 0.0, 0.0, 0};
      if (k < k1) {
        const int4 s = src[k];
        const int4 w4 = swin[k];
        en.xh = s.x;
        en.yh = s.y;
        en.xw = pairs ? w4.z : w4.x;  // 5w windows for collisions, boxes otherwise
        en.yw = pairs ? w4.w : w4.y;
        double f = gc.fluct ? (double)__int_as_float(s.z) : 1.0;
        double m = pairs ? gc.alpha : (ROOT ? 1.0 : gc.prefactor);
        if (pairs && gc.uli) {  // the pair's Gamma factor and (Alpha + (1 - Alpha) aw) of MCnucl.cpp:755
          const size_t pk = pbase + (size_t)(k - npart);
          f = gc.fluct ? (double)buf.pfluct[pk] : 1.0;
          m = gc.alpha + (1. - gc.alpha) * (double)buf.paw[pk];
        }
        const double fm = f * m;  // f gc.norm m as en.w + en.w_lo
        en.w = fm * gc.norm;
        en.w_lo = fma(fm, gc.norm, -en.w) + (fma(f, m, -fm) * gc.norm + fm * gc.norm_lo);
        const int xlo = en.xw & 0xffff, xhi = en.xw >> 16, ylo = en.yw & 0xffff, yhi = en.yw >> 16;
        if (xlo < xhi && ylo < yhi && ylo < c0 + kGY && yhi > c0)
#pragma unroll
          for (int v = 0; v < NW; ++v)
            if (xlo < R0 + TR * (v + 1) && xhi > R0 + TR * v) en.chunks |= 1 << v;
      }
      // ordered compaction: the tile's sources in list order
      const unsigned long long m = __ballot(en.chunks != 0);
      __syncthreads();  // the entries and counts of the last round are read
      if (lane == 0) cnt_s[wv] = __popcll(m);
      __syncthreads();
      int n = 0, at_n = 0;
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        if (v == wv) at_n = n;
        n += cnt_s[v];
      }
      if (en.chunks) wl[at_n + __popcll(m & ((1ull << lane) - 1ull))] = en;
      __syncthreads();
      for (int g = 0; g < n; g += kG64) {
        const int b = (g / kG64) & 1, ng = min(kG64, n - g);
        {  // rows of the 8 sources, then columns of 4 sources per pass
          const int s = t >> 5;
          if (s < ng) {
            const int xw = wl[g + s].xw;
            const double d = xg - (double)wl[g + s].xh * kH, d2 = d * d;
            const bool in = row >= (xw & 0xffff) && row < (xw >> 16);
            fx_s[b][s][fxi] = make_double2(in ? exp(-d2 / gc.two_w_w) : 0.0, d2);
          }
        }
#pragma unroll
        for (int p = 0; p < kG64; p += NW) {
          const int s = p + wv;
          if (s < ng) {
            const int yw = wl[g + s].yw;
            const double d = yg - (double)wl[g + s].yh * kH, d2 = d * d;
            const bool in = col >= (yw & 0xffff) && col < (yw >> 16);
            const double gy = exp(-d2 / gc.two_w_w);
            fy_s[b][s][lane] = make_double2(in ? fma(wl[g + s].w, gy, wl[g + s].w_lo * gy) : 0.0, d2);
          }
        }
        const int mine = g + (lane & (kG64 - 1));
        unsigned mm = (unsigned)__ballot(lane < ng && ((wl[mine].chunks >> wv) & 1));
        __syncthreads();
        while (mm) {
          const int u = __ffs((int)mm) - 1;
          mm &= mm - 1;
          double2 x[2], y[4];
#pragma unroll
          for (int i = 0; i < 2; ++i) x[i] = fx_s[b][u][TR * wv + 2 * q + i];
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) y[kk] = fy_s[b][u][16 * kk + c];
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
              if (x[i].y + y[kk].y <= cut) acc[i][kk] = fma(x[i].x, y[kk].x, acc[i][kk]);
        }
      }
    }
  }
  const size_t N = (size_t)cfg.nx * cfg.ny;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int ix = R0 + TR * wv + q + 4 * i;
    if (ix >= cfg.nx) continue;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int iy = c0 + c + 16 * k;
      if (iy < cfg.ny)
        out[(size_t)el * N + (size_t)ix * cfg.ny + iy] = ROOT ? sqrt(acc0[i][k] * acc[i][k]) : acc0[i][k] + acc[i][k];
    }
  }
}

int launch_grid64(const DevCfg& cfg, const EvBufs& b, const Grid64Const& gc, int ev0, int nev, double* out,
                  void* stream) {
  if (nev <= 0) return 0;
  const int ntx = (cfg.nx + kGX - 1) / kGX, nty = (cfg.ny + kGY - 1) / kGY;
  if (gc.model == 7)
    hipLaunchKernelGGL(k_grid64<true>, dim3(ntx * nty, nev), dim3(256), 0, (hipStream_t)stream, cfg, b, gc, ev0, out);
  else
    hipLaunchKernelGGL(k_grid64<false>, dim3(ntx * nty, nev), dim3(256), 0, (hipStream_t)stream, cfg, b, gc, ev0, out);
  return (int)hipGetLastError();
}

}  // namespace smc
