// Box flux tiles (box.h) of the persistent stage kernel (stage.hip): built with the FP
// contraction of fluxbox.hip and as relocatable device code, so its results are the bits of
// the separate launches.
#include "box.h"

namespace wmx {

template <int MODE, int SC>
__device__ void st_box(const StageStatic& s, const double* __restrict__ d_dt, double dt_host, int zfuse,
                       int tile) {
  box_tile<float, MODE, SC>(s.blks, s.tiles, s.ci_len, s.nd, s.pbuf[0], s.pbuf[1], s.pbuf[2], d_dt, dt_host, zfuse,
                            tile);
}

#define WMX_ST_BOX(C)                                                                  \
  template __device__ void st_box<1, C>(const StageStatic&, const double*, double, int, int); \
  template __device__ void st_box<2, C>(const StageStatic&, const double*, double, int, int); \
  template __device__ void st_box<3, C>(const StageStatic&, const double*, double, int, int);
WMX_ST_BOX(SC_ANY)
WMX_ST_BOX(SC_HYB_KEP4_ALBADA)
WMX_ST_BOX(SC_KEP2)
WMX_ST_BOX(SC_KEP4)
#undef WMX_ST_BOX

}  // namespace wmx
