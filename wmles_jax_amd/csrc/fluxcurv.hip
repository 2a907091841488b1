// Flux launches of curvilinear FP64 plans (curv.h) and the two metric planes they keep.
#include "curv.h"

namespace wmx {

// (FP64: 256 VGPRs, two workgroups per CU)
template <int MODE, int SC>
__global__ __launch_bounds__(256, 2) void k_curv(const BlockDev* __restrict__ blks, const int4* __restrict__ tiles,
                                                 int ci_len, NumDev nd, Ptrs qin, Ptrs q0, Ptrs out,
                                                 const double* __restrict__ d_dt, double dt_host, int zfuse) {
  curv_tile<MODE, SC>(blks, tiles, ci_len, nd, qin, q0, out, d_dt, dt_host, zfuse, (int)blockIdx.x);
}

hipError_t launch_curv(int mode, const BlockDev* d_blks, const int4* d_tiles, int ntiles, int ci_len,
                       const NumDev& nd, Ptrs qin, Ptrs q0, Ptrs out, const double* d_dt, double dt,
                       int zfuse, hipStream_t s) {
  if (ntiles <= 0) return hipSuccess;
  dim3 grid(ntiles), block(NT);
#define WMX_CV(M, C) hipLaunchKernelGGL((k_curv<M, C>), grid, block, 0, s, d_blks, d_tiles, ci_len, nd, qin, q0, out, d_dt, dt, zfuse)
#define WMX_CVM(C)               \
  switch (mode) {                \
    case 0: WMX_CV(0, C); break; \
    case 1: WMX_CV(1, C); break; \
    case 2: WMX_CV(2, C); break; \
    default: WMX_CV(3, C); break; \
  }
  switch (scheme_config(nd)) {
    case SC_HYB_KEP4_ALBADA: WMX_CVM(SC_HYB_KEP4_ALBADA); break;
    case SC_KEP2: WMX_CVM(SC_KEP2); break;
    case SC_KEP4: WMX_CVM(SC_KEP4); break;
    default: WMX_CVM(SC_ANY); break;
  }
#undef WMX_CVM
#undef WMX_CV
  return hipGetLastError();
}

// planes 0 and 1 of the record region: half the reciprocal volume and the filter width (a cube
// root) of every cell, made once at workspace binding
__global__ __launch_bounds__(256) void k_curv_geo(BlockDev B) {
  const unsigned c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= (unsigned)B.cells) return;
  const double v = B.vol[c];
  B.P[c] = 0.5 / v;
  B.P[(size_t)B.cells + c] = cbrt(v);
}

hipError_t launch_curv_geo(const BlockDev& hb, hipStream_t s) {
  hipLaunchKernelGGL(k_curv_geo, dim3((unsigned)((hb.cells + 255) / 256)), dim3(256), 0, s, hb);
  return hipGetLastError();
}

}  // namespace wmx
