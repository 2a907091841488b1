// Flux-kernel launches of unfused FP32-bulk plans: k_flux2 runs one marching tile per workgroup
// of the body in flux2.h.
#include "flux2.h"

namespace wmx {

// MODE 0: r = RHS; 1: q + dt r; 2: 3/4 q0 + 1/4 (q + dt r); 3: 1/3 q0 + 2/3 (q + dt r)
template <class R, int MODE, int SC>
__global__ __launch_bounds__(256, 2) void k_flux2(const BlockDev* __restrict__ blks,
                                               const int4* __restrict__ tiles, int ci_len,
                                               NumDev nd, Ptrs qin, Ptrs q0, Ptrs out,
                                               const double* __restrict__ d_dt, double dt_host) {
  flux2_tile<R, MODE, SC>(blks, tiles, ci_len, nd, qin, q0, out, d_dt, dt_host, (int)blockIdx.x);
}

// The Hybrid (KEP4 + MUSCL-HLLC) kernels are compiled in flux_ilp.hip (this file with
// WMX_FLUX_ILP_UNIT defined) under LLVM's max-ILP machine scheduler, which shortens them by
// 2-3% (the arithmetic is the same); the others, which it slows, are instantiated here by
// their launches.
#define WMX_FLUX_SIG (const BlockDev*, const int4*, int, NumDev, Ptrs, Ptrs, Ptrs, const double*, double)
#define WMX_FLUX_ILP_LIST(PFX)                                                   \
  PFX template __global__ void k_flux2<float, 0, SC_HYB_KEP4_ALBADA> WMX_FLUX_SIG; \
  PFX template __global__ void k_flux2<float, 1, SC_HYB_KEP4_ALBADA> WMX_FLUX_SIG; \
  PFX template __global__ void k_flux2<float, 2, SC_HYB_KEP4_ALBADA> WMX_FLUX_SIG; \
  PFX template __global__ void k_flux2<float, 3, SC_HYB_KEP4_ALBADA> WMX_FLUX_SIG;

#ifdef WMX_FLUX_ILP_UNIT
WMX_FLUX_ILP_LIST()
#else
WMX_FLUX_ILP_LIST(extern)


hipError_t launch_flux(int mode, const BlockDev* d_blks, const int4* d_tiles, int ntiles, int ci_len,
                       const NumDev& nd, Ptrs qin, Ptrs q0, Ptrs out, const double* d_dt,
                       double dt, hipStream_t s) {
  if (ntiles <= 0) return hipSuccess;
  dim3 grid(ntiles), block(NT);
#define WMX_F2(M, C) hipLaunchKernelGGL((k_flux2<float, M, C>), grid, block, 0, s, d_blks, d_tiles, ci_len, nd, qin, q0, out, d_dt, dt)
#define WMX_F2M(C)              \
  switch (mode) {               \
    case 0: WMX_F2(0, C); break; \
    case 1: WMX_F2(1, C); break; \
    case 2: WMX_F2(2, C); break; \
    default: WMX_F2(3, C); break; \
  }
  switch (scheme_config(nd)) {
    case SC_HYB_KEP4_ALBADA: WMX_F2M(SC_HYB_KEP4_ALBADA); break;
    case SC_KEP2: WMX_F2M(SC_KEP2); break;
    case SC_KEP4: WMX_F2M(SC_KEP4); break;
    default: WMX_F2M(SC_ANY); break;
  }
#undef WMX_F2M
#undef WMX_F2
  return hipGetLastError();
}
#endif

}  // namespace wmx
