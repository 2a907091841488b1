// Flux launches of box plans (box.h: every block's metrics are tensor products), and the
// tables and the check that make a block one.
#include "box.h"

namespace wmx {

// Occupancy: FP32 161 VGPRs and 52.9 KB of LDS, three workgroups per CU; FP64 256 VGPRs and
// 77 KB, two.  Measured per launch on the 256 x 128 x 128 channel (Hybrid KEP4 + MUSCL-HLLC,
// Vreman; events, mean of the stages): FP32 461 us + 78 us of primitive launch with the general
// fused kernel, 274 us here; FP64 920 us + 300 us of gradient launch + 137 us, 427 us here.  VALU
// issue and the latency of three dependent LDS phases per plane bound both; HBM does not.
template <class R, int MODE, int SC>
__global__ __launch_bounds__(256, sizeof(R) == 4 ? 3 : 2) void k_box(
    const BlockDev* __restrict__ blks, const int4* __restrict__ tiles, int ci_len, NumDev nd, Ptrs qin, Ptrs q0,
    Ptrs out, const double* __restrict__ d_dt, double dt_host, int zfuse) {
  box_tile<R, MODE, SC>(blks, tiles, ci_len, nd, qin, q0, out, d_dt, dt_host, zfuse, (int)blockIdx.x);
}

hipError_t launch_box(int mode, const BlockDev* d_blks, const int4* d_tiles, int ntiles, int ci_len,
                      const NumDev& nd, Ptrs qin, Ptrs q0, Ptrs out, const double* d_dt, double dt,
                      int zfuse, hipStream_t s) {
  if (ntiles <= 0) return hipSuccess;
  dim3 grid(ntiles), block(NT);
#define WMX_BX(R, M, C) hipLaunchKernelGGL((k_box<R, M, C>), grid, block, 0, s, d_blks, d_tiles, ci_len, nd, qin, q0, out, d_dt, dt, zfuse)
#define WMX_BXM(R, C)               \
  switch (mode) {                   \
    case 0: WMX_BX(R, 0, C); break; \
    case 1: WMX_BX(R, 1, C); break; \
    case 2: WMX_BX(R, 2, C); break; \
    default: WMX_BX(R, 3, C); break; \
  }
#define WMX_BXS(R)                                                      \
  switch (scheme_config(nd)) {                                          \
    case SC_HYB_KEP4_ALBADA: WMX_BXM(R, SC_HYB_KEP4_ALBADA); break;     \
    case SC_KEP2: WMX_BXM(R, SC_KEP2); break;                           \
    case SC_KEP4: WMX_BXM(R, SC_KEP4); break;                           \
    default: WMX_BXM(R, SC_ANY); break;                                 \
  }
  if (nd.prec == WMX_PREC_FP32_BULK) {
    WMX_BXS(float)
  } else {
    WMX_BXS(double)
  }
#undef WMX_BXS
#undef WMX_BXM
#undef WMX_BX
  return hipGetLastError();
}

// Tables of a block: along axis d the face coordinates of the line through the first interior
// cell of the other axes.
__global__ __launch_bounds__(256) void k_box_axes(BlockDev B) {
  const int d = blockIdx.y, x = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = B.N[d], ng = B.ng;
  if (x >= n) return;
  int c[3] = {ng, ng, ng};
  const double* xf = B.xf[d] + (size_t)d * fcount(B.N, d);
  const double* xc = B.xc + (size_t)d * B.cells;
  auto face = [&](int f) { c[d] = f; return xf[fidx(B.N, d, c[0], c[1], c[2])]; };
  auto centre = [&](int i) { c[d] = i; return xc[cidx(B.N, c[0], c[1], c[2])]; };
  BoxEnt e;
  e.w = face(x + 1) - face(x);
  e.iw = 1.0 / e.w;
  e.cb = cbrt(e.w);
  const double dist = x > 0 ? centre(x) - centre(x - 1) : 1.0;
  e.x = centre(x);
  e.id = 1.0 / fabs(dist);
  const float df = (float)dist;                  // as the FP32 faces form it
  e.idf = __builtin_amdgcn_rsqf(df * df);
  e.df = df;
  const_cast<BoxEnt*>(B.box[d])[x] = e;
}

// bad |= 1 unless every cell that a gradient record is formed for (the block's cells and one
// ghost layer) is a box of the tables: face vectors along their own axis only, and equal to
// the product of the two widths (1e-13: both are a few roundings of the same differences);
// the volume equal to the product of the three and the centroid to the table's, within tol of
// it.  The stored volume is a difference of coordinate-sized terms, whose rounding grows like
// |x| / width (7e-14 on the 256 x 128 x 128 channel, 1.3e-13 on 512 x 256 x 256; 3e-12 a
// thousand lengths from the origin), and the kernels divide by the product.  So tol is 4e-13
// for FP64 plans, which keeps their right-hand side within 1e-12 of one that divides by the
// stored volume, and 1e-11 for FP32-bulk plans, whose fluxes are 1e-7.  A NaN fails every
// comparison.
__global__ __launch_bounds__(256) void k_box_check(BlockDev B, double tol, unsigned* __restrict__ bad) {
  const int ng = B.ng;
  const int b1 = B.n[1] + 2, b2 = B.n[2] + 2;
  const long long l = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  bool ok = true;
  if (l < (long long)(B.n[0] + 2) * b1 * b2) {
    const int cc[3] = {ng - 1 + (int)(l / ((long long)b1 * b2)), ng - 1 + (int)((l / b2) % b1), ng - 1 + (int)(l % b2)};
    double w[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      w[d] = B.box[d][cc[d]].w;
      ok = ok && w[d] > 0.0;
    }
    const long long c = cidx(B.N, cc[0], cc[1], cc[2]);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double area = w[(d + 1) % 3] * w[(d + 2) % 3];
      const size_t fc = (size_t)fcount(B.N, d);
      for (int h = 0; h < 2; ++h) {
        int f[3] = {cc[0], cc[1], cc[2]};
        f[d] += h;
        const size_t fi = (size_t)fidx(B.N, d, f[0], f[1], f[2]);
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          const double S = B.S[d][x * fc + fi];
          ok = ok && (x == d ? fabs(S - area) <= 1e-13 * area : S == 0.0);
        }
      }
      ok = ok && fabs(B.xc[(size_t)d * B.cells + c] - B.box[d][cc[d]].x) <= tol * w[d];
    }
    const double vol = (w[0] * w[1]) * w[2];
    ok = ok && fabs(B.vol[c] - vol) <= tol * vol;
  }
  if (!__all(ok) && (threadIdx.x & 63) == 0 && *(volatile unsigned*)bad == 0u) atomicOr(bad, 1u);
}

hipError_t launch_box_check(const BlockDev& hb, int prec, unsigned* d_bad, hipStream_t s) {
  const int nmax = hb.N[0] > hb.N[1] ? (hb.N[0] > hb.N[2] ? hb.N[0] : hb.N[2]) : (hb.N[1] > hb.N[2] ? hb.N[1] : hb.N[2]);
  hipLaunchKernelGGL(k_box_axes, dim3((nmax + 255) / 256, 3), dim3(256), 0, s, hb);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const long long n = (long long)(hb.n[0] + 2) * (hb.n[1] + 2) * (hb.n[2] + 2);
  hipLaunchKernelGGL(k_box_check, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, hb,
                     prec == WMX_PREC_FP32_BULK ? 1e-11 : 4e-13, d_bad);
  return hipGetLastError();
}

}  // namespace wmx
